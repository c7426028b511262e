"""The bf16 score-tile kernels at p = 2 (fastmax_amd/csrc/fm_tiles.h) where they can go wrong -- edges of tiles, stages
and blocks, padded head dimensions, key prefixes, groups of heads, rows that start on odd addresses, coefficients small and
large against each other -- against the fp64 closed form.  Tolerance: bf16 rounds weights and outputs by at most 2^-9
each (3.9e-3 together); measured 2e-3 to 4e-3 normwise.  The largest difference is measured against the largest value, where
the first rows' sums of few terms round by up to 1e-2: the package's 2e-2 for bf16 inputs holds for both."""
import ctypes as C

import pytest
import torch

from oracle import fastmax_oracle as O

from helpers import TOL, assert_close

pytestmark = pytest.mark.gpu
KERNEL_PATH = "dense"


def check(bh, bhkv, nq, nk, d, mask, seed=0, scale=1.0, **kw):
    from fastmax_amd import ops

    print("tiles case", bh, bhkv, nq, nk, d, mask, kw, flush=True)
    kw = dict(dict(mask=mask, normalize=True, p=2), **kw)
    q, _, _, go = O.seeded_inputs((bh, nq, d), seed=seed, dtype=torch.bfloat16)
    _, k, v, _ = O.seeded_inputs((bhkv, nk, d), seed=seed + 1, dtype=torch.bfloat16)
    q, k = ((scale * t.float()).to(torch.bfloat16) for t in (q, k))
    qd, kd, vd, god = (t.cuda() for t in (q, k, v, go))
    o, den, sc, arg = ops.forward(qd, kd, vd, **kw)
    grads = ops.backward(qd, kd, vd, o, den, god, qk_scale=sc, qk_argmax=arg, **kw)
    r = bh // bhkv
    temp = kw.pop("temperature", 1.0)   # (divides the keys; only without normalisation)
    ref = O.dense_truth(q.float(), k.float().repeat_interleave(r, 0) / temp, v.float().repeat_interleave(r, 0), go.float(), **kw)
    fold = lambda t: t.reshape(bhkv, r, nk, d).sum(1)
    for name, got, want in zip(("o", "dq", "dk", "dv"), (o, *grads), (ref[0], ref[1], fold(ref[2]) / temp, fold(ref[3]))):
        assert_close(name, got.float(), want, TOL[torch.bfloat16], atol=1e-6)


@pytest.mark.parametrize("mask", [True, False])
@pytest.mark.parametrize("n,d", [(31, 64), (33, 8), (64, 128), (65, 24), (95, 96), (127, 32), (128, 104), (129, 64),
                                 (161, 40), (193, 72), (257, 128), (385, 64)])
def test_edges_of_tiles_and_head_dims(built, n, d, mask):
    check(2, 2, n, n, d, mask, seed=n + d)


@pytest.mark.parametrize("bh,bhkv,nq,nk,d,mask", [
    (3, 3, 2, 130, 64, True), (2, 2, 70, 333, 128, True), (2, 2, 129, 600, 32, True), (2, 2, 40, 150, 64, False), (2, 2, 200, 70, 96, False),
    (6, 2, 150, 150, 64, True), (8, 2, 129, 257, 128, True), (6, 1, 90, 90, 24, False), (600, 300, 70, 70, 64, True), (1100, 1100, 40, 40, 64, True),
    (4, 2, 65, 385, 128, True), (3, 1, 191, 191, 120, True), (580, 290, 65, 65, 128, True), (576, 288, 65, 65, 128, True),
    (260, 130, 33, 40, 128, False), (130, 65, 40, 130, 128, True), (256, 128, 130, 60, 128, False), (2, 2, 191, 191, 128, True)])
def test_prefixes_and_groups(built, bh, bhkv, nq, nk, d, mask):
    check(bh, bhkv, nq, nk, d, mask, seed=nq)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("a", [(1.0, -0.7, 0.3), (0.7, 1.3, -0.2), (0.0, 0.0, 1.0), (1.0, 0.0, 0.5), (1.0, 1.0, 1e-3), (1.0, 1.0, 9e-4)])
def test_coefficients(built, a, d):
    kw = dict(a0=a[0], a1=a[1], a2=a[2])
    if a[0] == 0.0:   # a denominator of squares: kept from zero by the number of keys
        check(2, 2, 300, 300, d, False, seed=7, **kw)
    else:
        check(2, 2, 150, 150, d, True, seed=8, **kw)
        check(2, 2, 150, 150, d, True, seed=9, scale=0.15, **dict(kw, normalize=False, temperature=1.7))


def test_a_group_with_a_scaleless_head(built):
    """A query head whose row norms overflow has scale 0: it attends evenly and adds nothing to dk, whatever the other heads
    of its group do."""
    from fastmax_amd import ops

    for d in (64, 128):
        for zero in (0, 1):
            q, k, v, go = (t.cuda() for t in O.seeded_inputs((2, 130, d), seed=d, dtype=torch.bfloat16))
            k, v = k[:1].contiguous(), v[:1].contiguous()
            q[zero, 5, :] = 1e30
            kw = dict(mask=True, normalize=True, p=2)
            o, den, sc, arg = ops.forward(q, k, v, **kw)
            assert sc[zero] == 0
            _, dk, dv = ops.backward(q, k, v, o, den, go, qk_scale=sc, qk_argmax=arg, **kw)
            other = 1 - zero
            o1, den1, sc1, arg1 = ops.forward(q[other:other + 1], k, v, **kw)
            _, dk1, _ = ops.backward(q[other:other + 1], k, v, o1, den1, go[other:other + 1], qk_scale=sc1, qk_argmax=arg1, **kw)
            assert_close("dk", dk.float(), dk1.float(), TOL[torch.bfloat16])
            mean = v.float().cumsum(1) / torch.arange(1, 131, device="cuda")[:, None]
            assert_close("o", o[zero].float(), mean[0], TOL[torch.bfloat16])
            assert torch.isfinite(dv.float()).all()


@pytest.mark.parametrize("d", [24, 64, 128])
def test_rows_of_o_on_odd_addresses(built, d):
    from fastmax_amd import _cabi, ops

    lib = _cabi.load()
    q, k, v, go = (t.cuda() for t in O.seeded_inputs((2, 100, d), seed=d, dtype=torch.bfloat16))
    kw = dict(mask=True, normalize=True, p=2)
    o, den, sc, arg = ops.forward(q, k, v, **kw)
    ds = _cabi.make_desc(2, 100, d, 1, True, True, 2)
    ws = torch.empty(lib.fastmax_workspace_bytes(C.byref(ds), _cabi.PASS_FORWARD), dtype=torch.uint8, device="cuda")
    wide = torch.full((2, 100, d + 1), 7.0, dtype=torch.bfloat16, device="cuda")
    _cabi.check(lib.fastmax_forward(C.byref(ds), q.data_ptr(), k.data_ptr(), v.data_ptr(), wide.data_ptr(), d + 1, den.data_ptr(), 1,
                                    None, None, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(wide[..., :d], o) and bool((wide[..., d] == 7.0).all())
    a = ops.backward(q, k, v, o, den, go, qk_scale=sc, qk_argmax=arg, **kw)
    b = ops.backward(q, k, v, wide, den, go, qk_scale=sc, qk_argmax=arg, **kw)
    assert all(torch.equal(x, y) for x, y in zip(a, b))


def normwise(bh, bhkv, nq, nk, d, mask, seed, scale=1.0, **kw):
    """Relative 2-norm errors of o, dq, dk, dv against the fp64 closed form."""
    from fastmax_amd import ops

    print("tiles errors", bh, bhkv, nq, nk, d, mask, kw, flush=True)
    kw = dict(dict(mask=mask, normalize=True, p=2), **kw)
    q, _, _, go = O.seeded_inputs((bh, nq, d), seed=seed, dtype=torch.bfloat16)
    _, k, v, _ = O.seeded_inputs((bhkv, nk, d), seed=seed + 1, dtype=torch.bfloat16)
    q, k = ((scale * t.float()).to(torch.bfloat16) for t in (q, k))
    qd, kd, vd, god = (t.cuda() for t in (q, k, v, go))
    o, den, sc, arg = ops.forward(qd, kd, vd, **kw)
    grads = ops.backward(qd, kd, vd, o, den, god, qk_scale=sc, qk_argmax=arg, **kw)
    r = bh // bhkv
    ref = O.dense_truth(q.float(), k.float().repeat_interleave(r, 0), v.float().repeat_interleave(r, 0), go.float(), **kw)
    fold = lambda t: t.reshape(bhkv, r, nk, d).sum(1)
    return {name: float((got.double().cpu() - want).norm() / want.norm())
            for name, got, want in zip(("o", "dq", "dk", "dv"), (o, *grads), (ref[0], ref[1], fold(ref[2]), fold(ref[3])))}


# A rounding to bf16 is off by at most 2^-9 = 2.0e-3 of a value and 1.1e-3 in the root mean square of many.  o takes two of them
# (weights, o), the gradients up to five (two operands, weights, the sum, what o carries over): 1.6e-3 and 2.5e-3.  Measured over
# these cases 1.9e-3 to 2.6e-3 and 2.5e-3 to 4.2e-3 (short sequences: few terms a sum); the bound is 5e-3.
NORMWISE = 5e-3


@pytest.mark.parametrize("bh,bhkv,n,d,mask", [(2, 2, 512, 64, True), (8, 2, 300, 128, True), (2, 2, 512, 96, False), (4, 1, 400, 32, True),
                                              (540, 540, 130, 64, True)])
def test_normwise_errors(built, bh, bhkv, n, d, mask):
    errors = normwise(bh, bhkv, n, n, d, mask, seed=d)
    assert max(errors.values()) <= NORMWISE, errors


@pytest.mark.parametrize("d", [24, 64, 96, 128])
@pytest.mark.parametrize("a0,a1,a2,lim", [(1e-2, 1.0, 1e-3, 0.1), (1e-3, 1.0, 1e-3, 0.05), (1e-4, 1.0, 1e-3, 0.01), (1e-4, 1.0, 1e-3, 0.03),
                                          (1e-6, 1.0, 0.5, 0.002)])
@pytest.mark.parametrize("mask", [True, False])
def test_small_constant_term(built, mask, a0, a1, a2, lim, d):
    """With normalised rows a weight is about a0 plus or minus lim^2 a1: where both are small against a1^2 / a2 it must still keep the
    8 bits bf16 has, as it does when f is formed from a0 up and would not as the difference of a square and a constant."""
    errors = normwise(2, 2, 512, 512, d, mask, seed=3, a0=a0, a1=a1, a2=a2, lim=lim)
    assert max(errors.values()) <= NORMWISE, errors


@pytest.mark.parametrize("d", [24, 64])
@pytest.mark.parametrize("a0,scale", [(1e-3, 0.01), (1e-4, 3e-3)])
def test_small_constant_term_and_small_rows(built, a0, scale, d):
    errors = normwise(2, 2, 512, 512, d, True, seed=3, scale=scale, normalize=False, a0=a0, a1=1.0, a2=1e-3)
    assert max(errors.values()) <= NORMWISE, errors


@pytest.mark.parametrize("mask", [True, False])
@pytest.mark.parametrize("d", [24, 64, 104, 128])
def test_an_infinity_in_the_last_row_stays_one(built, d, mask):
    """150 keys end within a stage: rows behind the last one count for nothing, also where the last one holds an infinity (times a
    weight of zero, a copy of it would make a NaN of the infinite sum)."""
    from fastmax_amd import ops

    print("tiles infinity in v", d, mask, flush=True)
    q, k, v, go = (t.cuda() for t in O.seeded_inputs((2, 150, d), seed=d, dtype=torch.bfloat16))
    v[0, -1, d - 1] = float("inf")
    o, den, *_ = ops.forward(q, k, v, mask=mask, normalize=True, p=2)
    sees = o[0, -1:] if mask else o[0]
    assert torch.all(sees[:, d - 1] == float("inf")) and torch.isfinite(sees[:, :d - 1]).all()
    assert torch.isfinite(o[1]).all() and torch.isfinite(den).all()


@pytest.mark.parametrize("mask", [True, False])
@pytest.mark.parametrize("d", [24, 40, 104])
def test_an_infinity_in_the_last_channel_stays_with_its_key(built, d, mask):
    """Head dimensions that are padded to a multiple of 32: an infinite key has infinite scores, and its queries an infinite
    denominator and no weight left for other keys, whose dv is finite."""
    from fastmax_amd import ops

    print("tiles infinity in k", d, mask, flush=True)
    q, k, v, go = (t.cuda() for t in O.seeded_inputs((2, 150, d), seed=d, dtype=torch.bfloat16))
    q, k = q * 0.2, k * 0.2
    k[0, 70, d - 1] = float("inf")
    kw = dict(mask=mask, normalize=False, p=2)
    o, den, sc, arg = ops.forward(q, k, v, **kw)
    first = 70 if mask else 0
    assert torch.all(den[0, first:] == float("inf")) and torch.isfinite(den[0, :first]).all() and torch.isfinite(den[1]).all()
    _, _, dv = ops.backward(q, k, v, o, den, go, qk_scale=sc, qk_argmax=arg, **kw)
    others = [j for j in range(150) if j != 70]
    assert torch.isfinite(dv[0, others]).all() and torch.isfinite(dv[1]).all()
