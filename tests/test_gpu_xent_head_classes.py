"""GPU parity of the classifier head at the sizes where it changes how it
reads W: 16 and 17 classes, a last class batch that is not full, K at 256 and
512 (one, two and four vectors a lane) and just past, K that leaves lanes
without a vector; against fp64, 1e-5 (as test_gpu_small_step.py)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,K,Cc", [(3, 4, 17), (5, 256, 17), (5, 260, 16), (16, 496, 27), (7, 512, 9), (7, 516, 31),
                                    (4, 1020, 5), (4, 1028, 32), (3, 2048, 1)])
def test_head_against_fp64(C, B, K, Cc):
    r = np.random.default_rng(B + K + Cc)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()  # noqa: E731
    h, W, b = r.standard_normal((B, K)), r.standard_normal((Cc, K)) / K ** 0.5, r.standard_normal(Cc)
    h, W, b = (a.astype(np.float32) for a in (h, W, b))
    S = np.maximum(r.standard_normal((B, K)), 0).astype(np.float32)
    lab = r.integers(0, Cc, B).astype(np.int32)
    lg, dl, dH, dX = (torch.empty(s, device="cuda") for s in ((B, Cc), (B, Cc), (B, K), (B, K)))
    am, rl = torch.empty(B, device="cuda", dtype=torch.int32), torch.empty(B, device="cuda")
    C.launch_by_id("xent_head_f32_v0", C.OpKind.XentHead, [t(h), t(W), t(b), torch.from_numpy(lab).cuda(), t(S)],
                   [lg, dl, am, rl, dH, dX])
    z = h.astype(np.float64) @ W.astype(np.float64).T + b
    e = np.exp(z - z.max(1, keepdims=True))
    d = e / e.sum(1, keepdims=True)
    d[np.arange(B), lab] -= 1.0
    d /= B
    dh = d @ W.astype(np.float64)
    # a single class has no gradient: compare against zero, not relative to it
    scale = lambda a: max(np.abs(a).max(), 1e-6)  # noqa: E731
    for got, want in ((lg, z), (dl, d), (dH, dh), (dX, dh * (S > 0))):
        assert np.abs(got.cpu().numpy() - want).max() / scale(want) < 1e-5
    assert np.array_equal(am.cpu().numpy(), z.argmax(1))
    row = np.log(e.sum(1)) + z.max(1) - z[np.arange(B), lab]
    assert np.abs(rl.cpu().numpy() - row).max() <= 1e-5 * max(np.abs(row).max(), 1.0)
