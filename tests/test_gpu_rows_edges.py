"""GPU parity of the row kernels at widths that are no register-resident
width of their own: one past and one short of each lane count's widest row,
rows that end inside a vector, and rows that start at any 4-byte alignment.
Against the fp64 oracle, normwise 1e-5 (fp32 sums of at most 32768 values);
row max and argmax exact.  The memory around the outputs is checked too.
"""
from __future__ import annotations

import struct

import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu

RRED = int.from_bytes(b"RRED", "little")
WIDTHS = [4, 5, 6, 7, 61, 63, 65, 127, 129, 255, 511, 513, 1000, 1023, 1025, 1537, 2047, 2049, 3073, 4095, 4097, 6143,
          6145, 8191, 8193, 10007, 10241, 12289, 16383, 16385, 20481, 24577, 32767]


def canvas(n, dtype=torch.float32, offset=0):
    """n elements at an element offset into memory filled with a marker."""
    t = torch.full((n + 64,), 77, device="cuda", dtype=dtype)
    return t, t[16 + offset:16 + offset + n]


def untouched(t, view):
    lo = view.storage_offset()
    return bool((t[:lo] == 77).all()) and bool((t[lo + view.numel():] == 77).all())


@pytest.mark.parametrize("cols", WIDTHS)
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_rows_of_any_width(C, cols, offset):
    R = 5 if cols < 200 else 3
    r = np.random.default_rng(cols * 4 + offset)
    x = (r.standard_normal((R, cols)) * 2 + 0.1).astype(np.float32)
    x[0] = -1e4
    x[1, -1] = x[1].max() + 1.0  # the maximum in the last column
    lab = r.integers(0, cols, R).astype(np.int32)
    lab[0], lab[1] = cols - 1, max(0, cols - 3)
    full, v = canvas(R * cols, offset=offset)
    v.copy_(torch.from_numpy(x).view(-1))
    tx = v.view(R, cols)
    yf, yv = canvas(R * cols, offset=offset)
    mx, sx = torch.empty(R, device="cuda"), torch.empty(R, device="cuda")
    C.op_call(C.OpKind.RowSoftmax, [tx], [yv.view(R, cols), mx, sx])
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    assert orc.rel_err(yv.view(R, cols).cpu().numpy(), e / e.sum(1, keepdims=True)) < 1e-5
    assert np.array_equal(mx.cpu().numpy(), x.max(1))
    assert orc.rel_err(sx.cpu().numpy(), x64.sum(1)) < 1e-5
    assert untouched(yf, yv)
    for op, ref in ((0, x64.sum(1)), (1, x64.max(1))):
        o = torch.empty(R, device="cuda")
        C.op_call(C.OpKind.RowReduce, [tx], [o], RRED, struct.pack("<i", op))
        assert orc.rel_err(o.cpu().numpy(), ref) < (1e-5 if op == 0 else 1e-30)
    loss, am, rl = torch.empty((), device="cuda"), torch.empty(R, device="cuda", dtype=torch.int32), torch.empty(
        R, device="cuda")
    df, dv = canvas(R * cols, offset=offset)
    C.op_call(C.OpKind.SoftmaxXent, [tx, torch.from_numpy(lab).cuda()], [loss, dv.view(R, cols), am, rl])
    row = np.log(e.sum(1)) + x64.max(1) - x64[np.arange(R), lab]
    d = e / e.sum(1, keepdims=True)
    d[np.arange(R), lab] -= 1.0
    assert np.array_equal(am.cpu().numpy(), x.argmax(1))
    assert orc.rel_err(rl.cpu().numpy(), row) < 1e-5
    assert abs(float(loss) - row.mean()) < 1e-5 * abs(row.mean())
    assert orc.rel_err(dv.view(R, cols).cpu().numpy(), d / R) < 1e-5
    assert untouched(df, dv) and untouched(full, v)
    # in place
    C.op_call(C.OpKind.RowSoftmax, [tx], [tx, mx, sx])
    assert torch.equal(v, yv) and untouched(full, v)


@pytest.mark.parametrize("cols", [5, 1000, 10007])
def test_rows_of_special_values(C, cols):
    x = torch.randn(6, cols, device="cuda")
    x[0] = -float("inf")
    x[1, :-1] = -float("inf")       # one finite value, in the last column
    x[2, cols // 2] = float("inf")
    x[3, 1] = float("nan")
    x[4] = torch.finfo(torch.float32).min
    y, mx = torch.empty_like(x), torch.empty(6, device="cuda")
    C.op_call(C.OpKind.RowSoftmax, [x], [y, mx])
    h = y.cpu()
    assert bool(torch.isnan(h[[0, 2, 3]]).all())
    assert h[1, -1] == 1.0 and bool((h[1, :-1] == 0).all())
    assert torch.allclose(h[4], torch.full((cols,), 1.0 / cols), rtol=1e-6)
    assert mx[0] == -float("inf") and mx[2] == float("inf") and mx[4] == torch.finfo(torch.float32).min
    lab = torch.tensor([0, cols - 1, 0, 0, cols, -1], device="cuda", dtype=torch.int32)
    loss, am, rl = torch.empty((), device="cuda"), torch.empty(6, device="cuda", dtype=torch.int32), torch.empty(
        6, device="cuda")
    C.op_call(C.OpKind.SoftmaxXent, [x, lab], [loss, y, am, rl])
    r = rl.cpu()
    assert r[1] == 0.0 and bool(torch.isnan(r[[0, 2, 3, 4, 5]]).all())  # 4, 5: labels out of range
    assert am[0] == 0 and am[1] == cols - 1 and am[2] == cols // 2 and am[4] == 0
    assert torch.allclose(y[4].cpu(), torch.full((cols,), 1.0 / cols / 6), rtol=1e-6)


@pytest.mark.parametrize("n", [1, 255, 257, 4096, 4097, 8200])
def test_loss_mean_of_many_rows(C, n):
    x = torch.randn(n, 64, device="cuda")
    lab = torch.randint(0, 64, (n,), device="cuda", dtype=torch.int32)
    loss, am, rl = torch.empty((), device="cuda"), torch.empty(n, device="cuda", dtype=torch.int32), torch.empty(
        n, device="cuda")
    C.op_call(C.OpKind.SoftmaxXent, [x, lab], [loss, torch.empty_like(x), am, rl])
    assert float(loss) == float(np.float32(rl.double().cpu().numpy().mean()))
