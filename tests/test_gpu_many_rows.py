"""GPU parity where a grid's lanes pass 2^32, which the runtime counts in 32
bits: every row must still be computed.  The rows repeat a short pattern, whose
result the fp64 oracle gives (fp32, normwise 1e-5); every repetition has the
pattern's own bits."""
from __future__ import annotations

import struct

import numpy as np
import pytest
import torch

import oracle as orc
from test_gpu_norm import BNEP, LNEP, dev, host, rng

pytestmark = pytest.mark.gpu

RRED = int.from_bytes(b"RRED", "little")


def repeated(pattern, times):
    return pattern.repeat(times, *([1] * (pattern.dim() - 1)))


def same(t, n):
    """Every n rows of t are its first n."""
    v = t.view(-1, n, *t.shape[1:])
    return all(bool((c == v[:1]).all()) for c in v.split(1 << 21))


@pytest.mark.parametrize("N", [3, 8])
@pytest.mark.parametrize("in_place", [False, True])
def test_layernorm_of_more_rows_than_a_grid(C, N, in_place):
    n, times = 8, (1 << 23) + 1  # 2^26 + 8 rows, 64 lanes each
    M = n * times
    r = rng(N)
    px, pdy = dev(r.standard_normal((n, N)) * 2 + 0.5, torch.float32), dev(r.standard_normal((n, N)), torch.float32)
    g, b = dev(r.standard_normal(N), torch.float32), dev(r.standard_normal(N), torch.float32)
    x, dy = repeated(px, times), repeated(pdy, times)
    mean, rstd = torch.zeros(M, device="cuda"), torch.zeros(M, device="cuda")
    y = x if in_place else torch.zeros_like(x)
    C.op_call(C.OpKind.LayerNormFwd, [x, g, b], [y, mean, rstd], LNEP, struct.pack("<f", 1e-5))
    y_ref, mu_ref, rs_ref = orc.layernorm_fwd_f64(host(px), host(g), host(b), eps=1e-5)
    for got, want in ((y, y_ref), (mean, mu_ref), (rstd, rs_ref)):
        assert orc.rel_err(host(got[:n]), want) < 1e-5 and same(got, n)
    x.copy_(repeated(px, times))
    dx_ref, dg_ref, db_ref = orc.layernorm_bwd_f64(host(px), host(pdy), mu_ref, rs_ref, host(g))
    for affine in (False, True):
        d = dy.clone()
        dx = d if in_place else torch.zeros_like(x)
        dg, db = torch.zeros(N, device="cuda"), torch.zeros(N, device="cuda")
        if affine:
            C.op_call(C.OpKind.LayerNormBwd, [x, d, g, mean, rstd], [dx, dg, db])
            assert orc.rel_err(host(dx[:n]), dx_ref) < 1e-5
            if N == 8:  # a lane adds up to 2^18 terms, each with an error of at most 2^-24 of the sum
                tol = 2.0 ** -6
                assert orc.rel_err(host(dg) / times, dg_ref) < tol and orc.rel_err(host(db) / times, db_ref) < tol
        else:
            C.op_call(C.OpKind.LayerNormBwd, [x, d, mean, rstd], [dx])
        assert same(dx, n)


@pytest.mark.parametrize("affine", [False, True])
def test_layernorm_of_no_rows_is_refused(C, affine):
    x, s, g = torch.empty((0, 8), device="cuda"), torch.empty(0, device="cuda"), torch.ones(8, device="cuda")
    with pytest.raises(RuntimeError, match="Internal"):
        if affine:
            C.op_call(C.OpKind.LayerNormBwd, [x, x, g, s, s],
                      [torch.empty_like(x), torch.empty(8, device="cuda"), torch.empty(8, device="cuda")])
        else:
            C.op_call(C.OpKind.LayerNormBwd, [x, x, s, s], [torch.empty_like(x)])


@pytest.mark.parametrize("n,times,cols", [(8, (1 << 21) + 1, 3), (16, (1 << 20) - 1, 5)])
def test_rows_of_more_than_a_grid(C, n, times, cols):
    """2^24 + 8 rows in the looping kernel (256 lanes each), and one launch's
    rows and a few in the register kernel."""
    R = n * times
    r = rng(cols)
    px = dev(r.standard_normal((n, cols)) * 2, torch.float32)
    plab = torch.from_numpy(r.integers(0, cols, n).astype(np.int32)).cuda()
    x, lab = repeated(px, times), repeated(plab, times)
    x64, l64 = host(px), plab.cpu().numpy()
    y, mx, sx = torch.zeros_like(x), torch.zeros(R, device="cuda"), torch.zeros(R, device="cuda")
    C.op_call(C.OpKind.RowSoftmax, [x], [y, mx, sx])
    e = np.exp(x64 - x64.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    for got, want in ((y, p), (mx, x64.max(1)), (sx, x64.sum(1))):
        assert orc.rel_err(host(got[:n]), want) < 1e-5 and same(got, n)
    for op, want in ((0, x64.sum(1)), (1, x64.max(1))):
        o = torch.zeros(R, device="cuda")
        C.op_call(C.OpKind.RowReduce, [x], [o], RRED, struct.pack("<i", op))
        assert orc.rel_err(host(o[:n]), want) < 1e-5 and same(o, n)
    loss, am, rl = torch.zeros((), device="cuda"), torch.zeros(R, device="cuda", dtype=torch.int32), torch.zeros(
        R, device="cuda")
    C.op_call(C.OpKind.SoftmaxXent, [x, lab], [loss, y, am, rl])
    row = np.log(e.sum(1)) + x64.max(1) - x64[np.arange(n), l64]
    d = p.copy()
    d[np.arange(n), l64] -= 1.0
    assert np.array_equal(am[:n].cpu().numpy(), x64.argmax(1)) and same(am, n)
    assert orc.rel_err(host(rl[:n]), row) < 1e-5 and same(rl, n)
    assert orc.rel_err(host(y[:n]), d / R) < 1e-5 and same(y, n)
    assert abs(float(loss) - row.mean()) < 1e-5 * abs(row.mean())


def test_batchnorm_of_more_channels_than_a_grid(C):
    """2^22 channels at 1024 lanes each, in place; all have the values -1 and
    +1 in turn, so that mean and variance are known."""
    n, Cc = 4099, (1 << 22) + 1
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("34 GB of channels")
    x = torch.empty((1, Cc, 1, n), device="cuda", dtype=torch.float16)
    x.view(Cc, n)[:, ::2] = -1
    x.view(Cc, n)[:, 1::2] = 1
    mu = -1 / n
    r = (1 - mu * mu + 1e-5) ** -0.5
    mean, rstd = torch.zeros(Cc, device="cuda"), torch.zeros(Cc, device="cuda")
    C.op_call(C.OpKind.BatchNormFwd, [x], [x, mean, rstd], BNEP, struct.pack("<fI", 1e-5, 0))
    assert float((mean - mu).abs().max()) < 1e-5 and float((rstd / r - 1).abs().max()) < 1e-5
    want = torch.full((n,), (1 - mu) * r, device="cuda")
    want[::2] = (-1 - mu) * r
    assert all(float((c.float() - want).abs().max()) < 2e-3 for c in x.view(Cc, n).split(1 << 18))
    del x
    torch.cuda.empty_cache()
