"""GPU test of how the FP16/FP32 LDS kernel stages x and takes its batches:
one batch (every batch length, rows that end inside it), two to several
batches with an odd and an even count, x in one and in several passes of the
workgroup, on small integers whose sums are exact in FP32."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from cudalab_amd.build import build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,per", [(torch.float16, 8), (torch.float32, 4)])
@pytest.mark.parametrize("chunks", [
    1, 16, 17, 33, 64, 65, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025,
    1537, 2047, 2049, 2560, 3073, 4094])
@pytest.mark.parametrize("n", [1, 9, 4096])
def test_batches_and_staging(dtype, per, chunks, n):
    ext, k = build("gemv"), chunks * per
    if n * k > 1 << 26:
        n = 300
    g = torch.Generator().manual_seed(chunks)
    W = torch.randint(-2, 3, (n, k), generator=g).to("cuda", dtype)
    x = torch.randint(-2, 3, (k,), generator=g).to("cuda", dtype)
    announce(f"gemv staging {dtype} n={n} k={k}")
    # products are at most 4 and |sum| <= 4 k < 2^24: exact in any order
    want = torch.mv(W.double(), x.double()).to(dtype)
    assert torch.equal(ext.forward("gemv_cdna4", W, x), want)
    assert torch.equal(ext.forward("gemv_lds_tiled", W, x), want)
