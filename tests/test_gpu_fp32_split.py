"""GPU parity of the fp32 path's fp16-split products (pieces of 4 blocks or
more) against the float64 closed form: the sizes around its blocks and head
tiles, and the inputs that leave its range and are run on fp32 MFMAs instead.

Tolerances are those of the fp32 path, 1e-4, in units of the largest value that
the output can take (the largest |C|): both paths round every product to
about 2^-23 of its size. Logits are kept to a few units, as there 1e-4 also
bounds what a rounding of the logit does to its weight.
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


# scales of C on both sides of the split's range (2^-10 .. 2^12 in the first
# block), with q scaled inversely so that the logits stay the same
@pytest.mark.parametrize("n_h", [16, 32])
@pytest.mark.parametrize("scale", [2.0 ** -40, 2.0 ** -13, 2.0 ** -12, 2.0 ** -9, 2.0 ** 8, 2.0 ** 9, 2.0 ** 11, 2.0 ** 30])
def test_scales(n_h, scale):
    q, c = _inputs(n_h, 200, 7)
    _check((q / np.float32(scale)).astype(np.float32), (c * np.float32(scale)).astype(np.float32), 1,
           f"n_h={n_h} scale={scale}")


# one token past the range after the first block (the piece is run again), in
# the first, and zero first blocks; several chunks, so that others stay split
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
