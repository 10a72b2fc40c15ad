"""GPU test of the workgroup-to-row mapping (xcd_block in cq_kernels.hip):
grids around the runs of 32 and 64 workgroups per XCD and their spans of 256
and 512, grids of a few workgroups, and partial last workgroups.  A mapping
that is not a bijection leaves rows unwritten or writes them twice with
another row's value; every row is checked against the oracle's exact value
(inputs on which every partial sum is exact), outputs prefilled with NaN."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from oracle import oracle as orc
from test_gpu_exact import _gemv_exact, _int4_exact, _np, _q8_exact, _same_bits

pytestmark = pytest.mark.gpu

GRIDS = (1, 7, 8, 9, 31, 255, 256, 257, 300, 511, 512, 513, 519, 767, 768, 1025)


@pytest.mark.parametrize("grid", GRIDS)
def test_every_row_once(ext4, ext8, cuda, grid):
    from cudalab_amd.build import build
    extg = build("gemv")
    for n in (4 * grid, 4 * grid - 3):          # four rows per 256-thread workgroup
        wq, s, x = _q8_exact(n, 1024, seed=n)
        want8 = orc.expect_exact_w8(_np(wq), _np(s), _np(x))
        for v in ("qgemv_cdna4", "qgemv_lds_tiled", "qgemv_baseline"):
            announce(f"qgemv map {v} n={n}")
            out = torch.full((n,), float("nan"), dtype=torch.float16, device="cuda")
            ext8.forward_into(v, wq, s, x, out)
            _same_bits(out, want8, f"{v} n={n}")
        wp, s4, x4 = _int4_exact(n, 4096, seed=n)
        want4 = orc.expect_exact_w4(_np(wp), _np(s4), _np(x4))
        for v in ("int4gemv_lds_r1", "int4gemv_lds_r2", "int4gemv_lds_tiled"):
            announce(f"int4gemv map {v} n={n}")
            out = torch.full((n,), float("nan"), dtype=torch.float16, device="cuda")
            ext4.forward_into(v, wp, s4, x4, out)
            _same_bits(out, want4, f"{v} n={n}")
        W, xg = _gemv_exact(n, 1000, torch.float16, seed=n)
        wantg = orc.expect_exact_gemv(_np(W), _np(xg))
        for v in ("gemv_cdna4", "gemv_lds_tiled"):
            announce(f"gemv map {v} n={n}")
            out = torch.full((n,), float("nan"), dtype=torch.float16, device="cuda")
            extg.forward_into(v, W, xg, out)
            _same_bits(out, wantg, f"{v} n={n}")
