"""GPU parity of the fp32 path's split products (chunks of 64 tokens or more:
operands as three bf16 parts each) against the float64 closed form: the sizes
around its blocks and head tiles, entries of very different size within a cache
(columns, tokens, scales up to the largest fp32 numbers), infinities.

Two tolerances. 1e-4 of the largest |C| is the fp32 path's own, for the cases
that only have to come out right. TOL_COLUMN is what fp32 products and sums
leave in each value column, however small the column, and would show a single
part or product of the split left out. Logits are kept to a few units, as there
it also bounds what a rounding of the logit does to its weight.
"""
import numpy as np
import pytest
import torch

from ada_mla import capi, synthetic
from oracle import mla_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _inputs(n_h, n, seed):
    return (synthetic.normal((n_h, 576), seed, np.float32), synthetic.normal((n, 576), seed + 1, np.float32))


def _run(q, c, splits):
    out = capi.decode_fused_fp32(torch.from_numpy(q).cuda(), torch.from_numpy(c).cuda(), num_splits=splits)
    torch.cuda.synchronize()
    return out.double().cpu().numpy()


def _check(q, c, splits, what):
    print(what, flush=True)
    got = _run(q, c, splits)
    want = O.closed_form(q.astype(np.float64), c.astype(np.float64))
    np.testing.assert_allclose(got, want, atol=TOL * np.abs(c[:, :512]).max(), rtol=TOL, err_msg=what)


# one chunk of 64 .. 145 tokens: 16-head workgroups below 128 tokens, 32-head
# ones from there on (where n_h allows); whole and ragged last blocks
@pytest.mark.parametrize("n_h", [16, 32, 48, 64])
@pytest.mark.parametrize("n", [63, 64, 65, 79, 112, 127, 128, 129, 144, 145, 300])
def test_sizes(n_h, n):
    q, c = _inputs(n_h, n, 100 + n)
    _check(q, c, 1, f"n_h={n_h} N={n}")


# scales of C, with q scaled inversely so that the logits stay the same
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("scale", [2.0 ** -40, 2.0 ** -13, 2.0 ** -12, 2.0 ** -9, 2.0 ** 8, 2.0 ** 9, 2.0 ** 11, 2.0 ** 30])
def test_scales(n_h, scale):
    q, c = _inputs(n_h, 200, 7)
    _check((q / np.float32(scale)).astype(np.float32), (c * np.float32(scale)).astype(np.float32), 1,
           f"n_h={n_h} scale={scale}")


# one large entry in the first block, a later one and the last, two chunks
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("row,value", [(3, 3e5), (100, 3e5), (399, 3e5), (250, 4e4)])
def test_one_large_token(n_h, row, value):
    q, c = _inputs(n_h, 400, 9)
    c[row, 5] = value
    q[:, 5] = 0  # its logit stays ordinary
    print(f"n_h={n_h} row={row} value={value}", flush=True)
    got = _run(q, c, 2)
    want = O.closed_form(q.astype(np.float64), c.astype(np.float64))
    keep = np.arange(512) != 5
    np.testing.assert_allclose(got[:, keep], want[:, keep], atol=TOL * 5, rtol=TOL)
    np.testing.assert_allclose(got[:, 5], want[:, 5], atol=TOL * value, rtol=TOL)


@pytest.mark.parametrize("n_h", [16, 32])
def test_zero_blocks_and_heads(n_h):
    q, c = _inputs(n_h, 300, 11)
    c[:40] = 0
    q[3] = 0
    q[5] *= np.float32(1e-30)
    _check(q, c, 1, f"zeros n_h={n_h}")


# columns of very different size: the rope part 2^-8 of the rest with a query 2^8 larger
@pytest.mark.parametrize("n_h", [16, 32])
def test_mixed_columns(n_h):
    q, c = _inputs(n_h, 300, 13)
    c[:, 512:] *= np.float32(2.0 ** -8)
    q[:, 512:] *= np.float32(2.0 ** 8)
    _check(q, c, 1, f"mixed n_h={n_h}")


# an infinity in a later block: heads whose logit it makes -inf give the token no
# weight and stay finite outside its column, as on fp32 MFMAs
@pytest.mark.parametrize("n_h", [16, 32])
def test_infinity(n_h):
    q, c = _inputs(n_h, 200, 15)
    c[150, 7] = np.inf
    print(f"inf n_h={n_h}", flush=True)
    got = _run(q, c, 1)
    neg = q[:, 7] < 0
    want = O.closed_form(q.astype(np.float64), np.delete(c, 150, 0).astype(np.float64))
    keep = np.arange(512) != 7
    np.testing.assert_allclose(got[neg][:, keep], want[neg][:, keep], atol=TOL * 5, rtol=TOL)
    assert np.isnan(got[neg][:, 7]).all() and np.isnan(got[~neg]).all()

# Relative 2-norm of a value column's error over the heads. The products are good
# to 2^-24, so it is the rounding of the fp32 sums: of the logits (partial sums
# of up to about 100 before the scale 1/sqrt(192), to 2^-18 each, a handful of
# them adding up like their square root: about 5e-7, a relative error of the
# weights) and of the outputs (2^-24 each). Measured 4e-7 .. 1e-6 here, up to
# 1.8e-6 on fp32 MFMAs. One of the six products of parts left out of either
# product gives 2.6e-6 (the third part of P) .. 1e-2 on test_columns' inputs
# (emulated in float64).
TOL_COLUMN = 2.5e-6


def _check_columns(q, c, splits, what, keep=slice(None)):
    print(what, flush=True)
    got = _run(q, c, splits)[:, keep]
    want = O.closed_form(q.astype(np.float64), c.astype(np.float64))[:, keep]
    err = np.linalg.norm(got - want, axis=0) / np.linalg.norm(want, axis=0)
    assert err.max() < TOL_COLUMN, f"{what}: column {err.argmax()}: {err.max():.2e}"


# sizes as above, 1 and several chunks: every column of ordinary inputs
@pytest.mark.parametrize("n_h", [16, 32, 48])
@pytest.mark.parametrize("n,splits", [(64, 1), (127, 1), (145, 1), (300, 1), (700, 5), (5000, 7)])
def test_columns(n_h, n, splits):
    q, c = _inputs(n_h, n, 200 + n)
    _check_columns(q, c, splits, f"n_h={n_h} N={n} splits={splits}")


# value columns far smaller than the rest: all of them, or a group, or every other
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("e", [16, 24, 28, 37, 60, 100])
@pytest.mark.parametrize("cols", [slice(0, 512), slice(100, 260), slice(1, 512, 2)])
def test_small_value_columns(n_h, e, cols):
    q, c = _inputs(n_h, 300, 17)
    c[:, cols] *= np.float32(2.0 ** -e)
    _check_columns(q, c, 1, f"n_h={n_h} e={e} {cols}")


# columns whose products carry the logits though their entries are far smaller
# than the others': the rope part, or some latent columns, 2^-e with a query 2^e larger
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("e", [8, 16, 18, 24, 28, 37, 60, 100])
@pytest.mark.parametrize("cols", [slice(512, 576), slice(30, 200)])
def test_small_columns_with_large_query(n_h, e, cols):
    q, c = _inputs(n_h, 300, 13)
    c[:, cols] *= np.float32(2.0 ** -e)
    q[:, cols] *= np.float32(2.0 ** e)
    _check_columns(q, c, 1, f"n_h={n_h} e={e} {cols}")


# tokens of ordinary size that get no weight (logits 140 below the others'),
# first, last or throughout, and the weight on tokens 2^-e as large
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("e", [16, 30, 60])
@pytest.mark.parametrize("rows", [slice(0, 40), slice(250, 300), slice(0, 300, 7)])
def test_small_tokens_carry_the_weight(n_h, e, rows):
    q, c = _inputs(n_h, 300, 19)
    q[:, 575] = 10
    c[:, 575] = 0
    big = c[rows].copy()
    big[:, 575] = -200
    c[:, :512] *= np.float32(2.0 ** -e)
    c[rows] = big
    _check_columns(q, c, 1, f"n_h={n_h} e={e} {rows}")


# every scale of the whole cache, with a query inversely as large
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("e", [-100, -60, -14, 14, 30, 60, 100])
def test_cache_scales(n_h, e):
    q, c = _inputs(n_h, 200, 7)
    _check_columns(q * np.float32(2.0 ** -e), c * np.float32(2.0 ** e), 1, f"n_h={n_h} e={e}")


# an entry near the largest fp32 number, in a value column that the query does
# not look at and in a rope column that takes the token's weight away
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("row", [3, 150, 199])
def test_largest_numbers(n_h, row):
    q, c = _inputs(n_h, 200, 21)
    c[row, 7] = 3.4e38
    q[:, 7] = 0
    _check_columns(q, c, 1, f"value n_h={n_h} row={row}")
    q, c = _inputs(n_h, 200, 21)
    c[row, 520] = 3.4e38
    q[:, 520] = -np.abs(q[:, 520])
    print(f"rope n_h={n_h} row={row}", flush=True)
    got = _run(q, c, 1)
    want = O.closed_form(q.astype(np.float64), np.delete(c, row, 0).astype(np.float64))
    err = np.linalg.norm(got - want, axis=0) / np.linalg.norm(want, axis=0)
    assert err.max() < TOL_COLUMN, f"{err.max():.2e}"


# an infinity in a rope column: a head whose logit it makes -inf gives the token
# no weight and is as if it were not there; the others have no value (inf - inf)
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("row", [3, 150, 199])
@pytest.mark.parametrize("value", [np.inf, -np.inf])
def test_infinite_rope_entry(n_h, row, value):
    q, c = _inputs(n_h, 200, 23)
    c[row, 540] = value
    print(f"n_h={n_h} row={row} value={value}", flush=True)
    got = _run(q, c, 1)
    none = q[:, 540] * np.sign(value) < 0
    want = O.closed_form(q[none].astype(np.float64), np.delete(c, row, 0).astype(np.float64))
    err = np.linalg.norm(got[none] - want, axis=0) / np.linalg.norm(want, axis=0)
    assert err.max() < TOL_COLUMN, f"{err.max():.2e}"
    assert np.isnan(got[~none]).all()


# a query entry near the largest fp32 number: the largest product takes all the weight
@pytest.mark.parametrize("n_h", [16, 32])
def test_largest_query(n_h):
    q, c = _inputs(n_h, 200, 25)
    q[:, 530] = np.copysign(np.float32(3.4e38), q[:, 530])
    c[:, 530] *= np.float32(2.0 ** -100)
    _check_columns(q, c, 1, f"n_h={n_h}")
