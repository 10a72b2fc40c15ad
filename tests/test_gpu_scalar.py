"""GPU tests of the scalar kernels (the *_baseline variants and every call
off the vector contract) where their plan changes form: one, two or four
waves per row (1, 2-3, 4+ rounds of 64 chunks), one or two chunks per batch
(16+ rounds), one or two rows per wave (512 / 513 rows), rows shorter than
one chunk, and every length of the last, partial chunk.  Inputs on which
every partial sum is exact (test_gpu_exact.py), so any order of the sums
gives the oracle's value bit for bit; operands at several offsets.
"""
from __future__ import annotations

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


# whole chunks of a row, none a multiple of 64, so that lanes of the last round
# re-read the row's last chunk: one wave per row; two; four; four with batches
# of two chunks, whose last batch passes the wave's last round
PART_ROUNDS = (40, 72, 136, 324, 1028, 1156, 2116)


def _signs(like):
    """+1, -1, +1, ... down the rows."""
    return torch.tensor([1, -1] * 4, device="cuda").to(like)


@pytest.mark.parametrize("chunks", PART_ROUNDS)
@pytest.mark.parametrize("per", [32, 16, 8, 4], ids=["int4", "int8", "f16", "f32"])
def test_scalar_nonfinite(ext4, ext8, cuda, per, chunks):
    """Rounds that re-read a row's last chunk add nothing of it, whichever of
    its operands is infinite: a zero in the place of the other one would make
    the row NaN instead of +-Inf.  A NaN stays in its own row."""
    from cudalab_amd.build import build
    inf, nan, n = float("inf"), float("nan"), 8
    assert chunks % 64
    k = chunks * per
    last = k - per                       # the last whole chunk starts here
    x = torch.ones(k, dtype=torch.float32 if per == 4 else torch.float16, device="cuda")
    xi = x.clone()
    xi[last + 1] = inf
    want = inf * _signs(torch.float32)
    if per == 32:
        # weights +1 (0x11) or -1 (0xFF) by row; the last group's scale infinite
        W = torch.where(_signs(torch.float32) > 0, 0x11, 0xFF).to(torch.uint8)
        W = W.unsqueeze(1).repeat(1, k // 2)
        s = torch.full((n, k // 128), 0.25, dtype=torch.float16, device="cuda")
        si, sn = s.clone(), s.clone()
        si[:, -1], sn[3, -1] = inf, nan
        calls = {"x": (W, s, xi), "scale": (W, si, x), "nan": (W, sn, x)}
        run = lambda *a: ext4.forward("int4gemv_baseline", *a)     # noqa: E731
    elif per == 16:
        W = _signs(torch.int8).unsqueeze(1).repeat(1, k)
        s = torch.full((n,), 0.25, device="cuda")
        sn = s.clone()
        sn[3] = nan
        calls = {"x": (W, s, xi), "scale": (W, torch.full_like(s, inf), x), "nan": (W, sn, x)}
        run = lambda *a: ext8.forward("qgemv_baseline", *a)        # noqa: E731
    else:
        W = (0.25 * _signs(x.dtype)).unsqueeze(1).repeat(1, k)
        Wi, Wn = W.clone(), W.clone()
        Wi[:, last + 1] = inf * _signs(x.dtype)
        Wn[3, last + 1] = nan
        calls = {"x": (W, xi), "W": (Wi, x), "nan": (Wn, x)}
        run = lambda *a: build("gemv").forward("gemv_baseline", *a)  # noqa: E731
    for what, args in calls.items():
        announce(f"scalar non-finite {what} per={per} k={k}")
        y = run(*args).float()
        if what == "nan":
            finite = (0.25 * k * _signs(torch.float32)).to(x.dtype).float()
            assert torch.isnan(y[3]) and torch.equal(y[:3], finite[:3]) \
                and torch.equal(y[4:], finite[4:]), (what, y)
        else:
            assert torch.equal(y, want), (what, y)
