"""GPU tests of infinite operands in the vector kernels.  Lanes past the row
end re-read the row's last chunk of W and sum nothing of it: an Inf there
(FP16/FP32 W) or in x meets only its own product, and the row is +-Inf as on
the scalar kernel, not NaN (0 * Inf).  Chunk counts that leave lanes, chunks of
a lane or both past the row end, in one batch, in the last of several, and in
the last tile; full rows beside them."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from cudalab_amd.build import build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,per", [(torch.float16, 8), (torch.float32, 4)],
                         ids=["f16", "f32"])
@pytest.mark.parametrize("chunks", [1, 9, 16, 17, 33, 64, 65, 128, 129, 200, 257, 320, 511,
                                    512, 513, 1023, 1025, 1376, 2048, 2049, 2600, 4097, 4700])
def test_infinite_operands(cuda, dtype, per, chunks):
    ext, k, n = build("gemv"), chunks * per, 12
    inf = float("inf")
    W = torch.full((n, k), 0.25, dtype=dtype, device="cuda")
    x = torch.ones(k, dtype=dtype, device="cuda")
    # rows 0, 3, 6, 9 hold +Inf, 1, 4, 7, 10 -Inf, the others neither
    want = torch.tensor([inf, -inf, k / 4] * 4, dtype=dtype, device="cuda")
    for at in (k - 1, k - per, 0):      # ends of the last chunk, the row's start
        Wi = W.clone()
        Wi[0::3, at], Wi[1::3, at] = inf, -inf
        for v in ("gemv_cdna4", "gemv_lds_tiled", "gemv_baseline"):
            announce(f"gemv inf W {v} {dtype} k={k} at {at}")
            y = ext.forward(v, Wi, x)
            assert torch.equal(y, want), (v, at, y)
    x[k - 1] = inf
    Ws = W.clone()
    Ws[1::2] = -0.25
    want = torch.tensor([inf, -inf] * (n // 2), dtype=dtype, device="cuda")
    for v in ("gemv_cdna4", "gemv_lds_tiled", "gemv_baseline"):
        announce(f"gemv inf x {v} {dtype} k={k}")
        assert torch.equal(ext.forward(v, Ws, x), want), v


@pytest.mark.parametrize("k", [128, 256, 640, 2048, 2176, 4096, 11008, 16384, 16512, 28672, 35072])
@pytest.mark.parametrize("op", ["int4gemv", "qgemv"])
def test_infinite_x_of_quantized_weights(cuda, op, k):
    ext, n = build(op), 12
    sign = torch.tensor([1, -1] * (n // 2), device="cuda")
    if op == "int4gemv":
        W = torch.where(sign > 0, 0x11, 0xFF).to(torch.uint8).unsqueeze(1).repeat(1, k // 2)
        s = torch.full((n, k // 128), 0.25, dtype=torch.float16, device="cuda")
    else:
        W = sign.to(torch.int8).unsqueeze(1).repeat(1, k)
        s = torch.full((n,), 0.25, device="cuda")
    want = (float("inf") * sign).half()
    for at in (0, k - 1):
        x = torch.ones(k, dtype=torch.float16, device="cuda")
        x[at] = float("inf")
        for v in ext.variants():
            announce(f"{op} inf x {v} k={k} at {at}")
            assert torch.equal(ext.forward(v, W, s, x), want), (v, at)
