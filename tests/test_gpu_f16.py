"""fp16 conversions of the kernels, every f16 value, against numpy (exact)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
F16 = torch.float16


def test_f16_conversions_every_value(C):
    """f16 -> fp32 of every bit pattern, and fp32 -> f16 (RNE, overflow,
    subnormals, infinities, one NaN) of their pairwise sums, through the
    column sum."""
    bits = np.arange(65536, dtype=np.uint16)
    x = torch.from_numpy(bits.view(np.int16)).view(F16).cuda().view(1, -1)
    o = torch.empty(65536, device="cuda")
    C.op_call(C.OpKind.ReduceSum, [x], [o])
    f = bits.view(np.float16).astype(np.float32)
    assert np.array_equal(o.cpu().numpy(), f, equal_nan=True)
    for shift in (1, 77, 1024, 5000, 31744, 32768, 40000):
        other = np.roll(bits, shift)
        two = torch.from_numpy(np.stack([bits, other]).view(np.int16)).view(F16).cuda()
        oh = torch.empty(65536, device="cuda", dtype=F16)
        C.op_call(C.OpKind.ReduceSum, [two], [oh])
        with np.errstate(all="ignore"):
            want = (f + other.view(np.float16).astype(np.float32)).astype(np.float16)
        got = oh.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        # -0 + -0 may come out as +0 (the sum starts at +0)
        assert np.array_equal(got[ok], want[ok])
        assert np.all((got.view(np.uint16)[~ok] & 0x7fff) == 0x7e00)
