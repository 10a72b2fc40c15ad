"""GPU test of the INT8 quantizer's row splits (one, two, four or eight waves
per row, one to eight held chunks per thread, rows past what is held) and of
partial last workgroups, bit for bit against the oracle's quantizer; and of
the INT4 quantizer where its last workgroup is partial and its output is only
4-byte aligned."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _weights(n, k, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(n, k, generator=g) * 0.05).half()


# chunks of 8 per row around each change of the split: 64 (H 1/2), 128, 192,
# 256, 384, 512, 768, 1024, 1536, 2048, 4096 chunks
@pytest.mark.parametrize("chunks", [1, 63, 64, 65, 128, 129, 192, 193, 256, 257, 384,
                                    385, 512, 513, 768, 769, 1024, 1025, 1536, 1537,
                                    2048, 2049, 4096, 4097])
def test_q8_row_splits(cuda, chunks):
    from cudalab_amd.ext import quantize_q8, quantize_vectorized
    for n in (1, 3, 9):
        W = _weights(n, 8 * chunks, seed=chunks + n)
        W[n // 2, -1] = 3.0             # the row's amax in its last element
        announce(f"int8 quantize split n={n} chunks={chunks}")
        Wd = W.cuda()
        wq, s = quantize_q8(Wd)
        assert quantize_vectorized("qgemv", Wd, wq)
        owq, os_ = orc.quantize_w8_c(W.numpy(), rcp=True)
        assert np.array_equal(wq.cpu().numpy(), owq)
        assert np.array_equal(s.cpu().numpy().view(np.uint32), os_.view(np.uint32))


@pytest.mark.parametrize("n,k", [(1, 128), (31, 128), (32, 128), (33, 128), (7, 1152)])
def test_int4_partial_workgroups(cuda, n, k):
    from cudalab_amd import _capi
    lib = _capi.load()
    W = _weights(n, k, seed=n + k)
    Wd = W.cuda()
    owp, os_ = orc.quantize_w4_c(W.numpy(), rcp=True)
    for off in (0, 4, 8):               # wp 4-byte aligned is enough
        buf = torch.full((n * k // 2 + 32,), 0x5A, dtype=torch.uint8, device="cuda")
        wp = buf[off:off + n * k // 2]
        s = torch.empty(n, k // 128, dtype=torch.float16, device="cuda")
        announce(f"int4 quantize n={n} k={k} out+{off}")
        assert lib.cq_quantize_vectorized(0, Wd.data_ptr(), wp.data_ptr(), n, k) == 1
        assert lib.cq_int4_quantize(Wd.data_ptr(), wp.data_ptr(), s.data_ptr(), n, k, 1,
                                    torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        assert np.array_equal(wp.cpu().numpy().reshape(n, -1), owp)
        assert np.array_equal(s.cpu().numpy().view(np.uint16), os_.view(np.uint16))
        rest = torch.cat([buf[:off], buf[off + n * k // 2:]])
        assert bool((rest == 0x5A).all())


@pytest.mark.parametrize("op,shape,w_off", [
    ("int4gemv", (40, 384), 0), ("int4gemv", (40, 384), 2),
    ("qgemv", (9, 520), 0), ("qgemv", (9, 2056), 0), ("qgemv", (9, 2056), 2),
    ("qgemv", (9, 513), 0), ("qgemv", (3, 40000), 0)])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan"), 65504.0])
def test_nonfinite_word(cuda, op, shape, w_off, bad):
    """One NaN or Inf anywhere sets the word on every kernel (vectorized,
    element-wise, longer than held); the largest finite value does not, and
    neither does an earlier call's finding."""
    from cudalab_amd.ext import quantize_finite
    n, k = shape
    buf = torch.empty(n * k + 8, dtype=torch.float16, device="cuda")
    W = buf[w_off // 2:w_off // 2 + n * k].view(n, k)
    for pos in ((0, 0), (n - 1, k - 1), (n // 2, k // 3)):
        W.copy_(_weights(n, k, seed=1))
        announce(f"{op} nonfinite {bad} at {pos} of {shape} w+{w_off}")
        W[pos] = bad
        assert quantize_finite(op, W)[2] == (bad == 65504.0)
        W[pos] = 0.0
        assert quantize_finite(op, W)[2]
