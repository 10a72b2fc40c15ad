"""GPU test of grouped calls that also write one output with its runs
repeated (forward_grouped_repeat): inside the grouped launch (up to three
problems with one x, a power-of-two run) and by a copy behind it (an x each,
four problems, other runs, the K-tiled and the scalar kernels), through the
fast and the checked path; and of what is refused."""
from __future__ import annotations

import pytest
import torch

from conftest import announce
from test_gpu_exact import _int4_exact, _q8_exact

pytestmark = pytest.mark.gpu


def _repeat(y, head, times):
    return y.view(-1, 1, head).expand(-1, times, head).reshape(-1)


@pytest.mark.parametrize("op", ["int4gemv", "qgemv"])
@pytest.mark.parametrize("K,rows,index,head,shared", [
    (1024, (300, 256, 256), 2, 128, True), (4096, (256,), 0, 128, True),
    (4096, (1, 384), 1, 128, True), (1024, (384, 33), 0, 1, True),
    (1024, (8, 513), 0, 8, True), (2048, (64, 256, 3), 1, 256, True),
    (1024, (300, 256, 256), 1, 128, False), (1024, (7, 256, 9, 33), 1, 128, True),
    (1024, (300, 96), 1, 48, True), (16512, (33, 256), 1, 128, True)])
def test_repeated_output(ext4, ext8, monkeypatch, op, K, rows, index, head, shared):
    ext, make = (ext4, _int4_exact) if op == "int4gemv" else (ext8, _q8_exact)
    probs = [make(n, K, seed=3 * i + n) for i, n in enumerate(rows)]
    if shared:
        probs = [(W, s, probs[0][2]) for W, s, _ in probs]
    for variant in (f"{op}_cdna4", f"{op}_baseline"):
        want = [ext.forward(variant, *p) for p in probs]
        for times, checked in ((1, False), (2, False), (8, False), (3, True)):
            announce(f"{variant} repeat K={K} rows={rows} x{times} checked={checked}")
            outs = [torch.full_like(w, float("nan")) for w in want]
            rep = torch.full((rows[index] * times,), float("nan"), dtype=torch.float16,
                             device="cuda")
            problems = [(*p, o) for p, o in zip(probs, outs)]
            # an iterator is left to the checked path
            ext.forward_grouped_repeat(variant, iter(problems) if checked else problems,
                                       index, rep, head)
            for o, w in zip(outs, want):
                assert torch.equal(o, w)
            assert torch.equal(rep, _repeat(want[index], head, times))


def test_refused(ext4):
    W, s, x = _int4_exact(256, 1024, seed=1)
    out = torch.zeros(256, dtype=torch.float16, device="cuda")
    rep = torch.zeros(512, dtype=torch.float16, device="cuda")
    go = lambda *a: ext4.forward_grouped_repeat("int4gemv_cdna4", [(W, s, x, out)], *a)  # noqa: E731
    for args, what in (((1, rep, 128), "names no problem"), ((0, rep, 100), "runs of 100"),
                       ((0, rep[:300], 128), "300 elements"), ((0, rep.float(), 128), "float16"),
                       ((0, rep[::2], 128), "contiguous"), ((0, rep.view(2, 256), 128), "1-D")):
        with pytest.raises(RuntimeError, match=what):
            go(*args)
    both = torch.zeros(600, dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="overlaps an operand"):
        ext4.forward_grouped_repeat("int4gemv_cdna4", [(W, s, x, both[:256])], 0,
                                    both[88:], 128)
    torch.cuda.synchronize()
    assert not out.any() and not rep.any() and not both.any()
