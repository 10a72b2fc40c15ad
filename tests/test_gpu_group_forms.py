"""GPU test of the two grouped kernels: up to three problems with one x, and
any other group of up to eight.  Every output must equal the single call's
bit for bit: counts 1 to 8, one x or one per problem, problems of one row and
of partial last workgroups, rows of 16, 32 and 64 lanes and of one to several
chunks per lane, requested rows per lane."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from test_gpu_exact import _int4_exact, _q8_exact

pytestmark = pytest.mark.gpu

ROWS = (300, 1, 4099, 33, 64, 513, 7, 2048)


@pytest.mark.parametrize("K", [128, 1024, 2048, 4096, 6144, 16384])
@pytest.mark.parametrize("shared", [True, False], ids=["one-x", "own-x"])
@pytest.mark.parametrize("op", ["int4gemv", "qgemv"])
def test_grouped_equals_single(ext4, ext8, op, shared, K):
    ext, make = (ext4, _int4_exact) if op == "int4gemv" else (ext8, _q8_exact)
    probs = [make(n, K, seed=10 * i + n) for i, n in enumerate(ROWS)]
    # weights and x of ordinary values: the bits then depend on every sum's order
    g = torch.Generator(device="cuda").manual_seed(K)
    xs = [torch.randn(K, device="cuda", generator=g).half() for _ in ROWS]
    probs = [(W, s, xs[0] if shared else x) for (W, s, _), x in zip(probs, xs)]
    for variant in (f"{op}_cdna4", f"{op}_lds_r2"):
        want = [ext.forward(variant, *p) for p in probs]
        for count in (1, 2, 3, 4, 8):
            for first in range(0, len(probs) - count + 1, 2):
                part = probs[first:first + count]
                outs = [torch.full((p[0].size(0),), float("nan"), dtype=torch.float16,
                                   device="cuda") for p in part]
                announce(f"{variant} group K={K} shared={shared} [{first}:{first + count}]")
                ext.forward_grouped(variant, [(*p, o) for p, o in zip(part, outs)])
                for i, o in enumerate(outs):
                    assert torch.equal(o.view(torch.int16),
                                       want[first + i].view(torch.int16)), (count, first, i)
