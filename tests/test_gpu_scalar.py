"""GPU tests of the scalar kernels (the *_baseline variants and every call
off the vector contract) where their plan changes form: one, two or four
waves per row (1, 2-3, 4+ rounds of 64 chunks), one or two chunks per batch
(16+ rounds), one or two rows per wave (512 / 513 rows), rows shorter than
one chunk, and every length of the last, partial chunk.  Inputs on which
every partial sum is exact (test_gpu_exact.py), so any order of the sums
gives the oracle's value bit for bit; operands at several offsets.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import oracle as orc
from test_gpu_exact import (_gemv_exact, _int4_exact, _misaligned, _np, _q8_exact,
                            _same_bits)

pytestmark = pytest.mark.gpu

ROWS = (1, 5, 512, 513)


def _lengths(per):
    """Row lengths around each boundary of the plan, for `per` elements a
    chunk: below one chunk, and 1..17 rounds of 64 chunks with a remainder."""
    step = 64 * per
    out = [1, per - 1, per, per + 1, step - 1, step, step + 3]
    for rounds in (2, 3, 4, 15, 16, 17, 33):
        out += [rounds * step - per + 1, rounds * step, rounds * step + 1]
    return out


@pytest.mark.parametrize("k", sorted(set(_lengths(16))))
def test_q8_scalar_exact(ext8, k):
    for n in ROWS:
        wq, s, x = _q8_exact(n, k, seed=n + k)
        want = orc.expect_exact_w8(_np(wq), _np(s), _np(x))
        for woff, xoff in ((0, 0), (1, 2), (6, 14)):
            announce(f"qgemv scalar n={n} k={k} w+{woff} x+{xoff}")
            y = ext8.forward("qgemv_baseline", _misaligned(wq, woff), s, _misaligned(x, xoff))
            _same_bits(y, want, f"n={n} k={k} w+{woff} x+{xoff}")


@pytest.mark.parametrize("dtype,per", [(torch.float16, 8), (torch.float32, 4)],
                         ids=["f16", "f32"])
def test_gemv_scalar_exact(cuda, dtype, per):
    from cudalab_amd.build import build
    extg = build("gemv")
    es = 16 // per
    for k in sorted(set(_lengths(per))):
        for n in ROWS:
            W, x = _gemv_exact(n, k, dtype, seed=n + k)
            want = orc.expect_exact_gemv(_np(W), _np(x))
            announce(f"gemv scalar {dtype} n={n} k={k}")
            for woff, xoff in ((0, 0), (es, es), (3 * es, 0)):
                y = extg.forward("gemv_baseline", _misaligned(W, woff), _misaligned(x, xoff))
                _same_bits(y, want, f"{dtype} n={n} k={k} w+{woff} x+{xoff}")


@pytest.mark.parametrize("k", [128, 2048, 2176, 4096, 6144, 6272, 8192, 8320,
                               30720, 32768, 32896, 65536])
def test_int4_scalar_exact(ext4, k):
    for n in ROWS:
        wp, s, x = _int4_exact(n, k, seed=n + k)
        want = orc.expect_exact_w4(_np(wp), _np(s), _np(x))
        for woff, xoff in ((0, 0), (1, 2), (7, 14)):
            announce(f"int4gemv scalar n={n} k={k} w+{woff} x+{xoff}")
            y = ext4.forward("int4gemv_baseline", _misaligned(wp, woff), s, _misaligned(x, xoff))
            _same_bits(y, want, f"n={n} k={k} w+{woff} x+{xoff}")


def test_scalar_nonfinite(ext8, cuda):
    """Inf and NaN operands meet exactly their own products: the rounds that
    re-read a row's last chunk add nothing."""
    from cudalab_amd.build import build
    k = 64 * 16 + 5
    wq, s, x = _q8_exact(8, k, seed=3)
    wq[wq == 0] = 1
    x.fill_(1.0)
    x[k - 1] = float("inf")             # in the partial chunk
    wq[:, k - 1] = torch.tensor([1, -1] * 4, dtype=torch.int8, device="cuda")
    announce("qgemv scalar inf x")
    y = ext8.forward("qgemv_baseline", wq, s, x)
    assert torch.equal(y, torch.tensor([np.inf, -np.inf] * 4, device="cuda").half())
    extg = build("gemv")
    W = torch.ones(8, k, dtype=torch.float16, device="cuda")
    W[:, 64 * 16 - 1] = float("inf")    # last element of the last whole chunk
    announce("gemv scalar inf W")
    y = extg.forward("gemv_baseline", W, torch.ones(k, dtype=torch.float16, device="cuda"))
    assert torch.isposinf(y).all()
