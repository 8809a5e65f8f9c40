"""GPU parity of LayerNorm and BatchNorm with every tensor at an odd element
address inside memory filled with a marker that must survive: unaligned vector
loads and stores, vectors moved back to a row's end, and the partial sums that
the fused LayerNorm backward and the split BatchNorm keep in dx or y at an
address rounded up.  Oracle and tolerances as in test_gpu_norm.py."""
from __future__ import annotations

import struct

import pytest
import torch

import oracle as orc
from test_gpu_norm import BNEP, LNEP, host, rng

pytestmark = pytest.mark.gpu

F32, F16 = torch.float32, torch.float16
MARK = 77.0


class Canvas:
    """Views at an element offset into marked memory."""

    def __init__(self, offset):
        self.offset, self.made = offset, []

    def view(self, shape, dtype, values=None):
        n = int(torch.Size(shape).numel())
        full = torch.full((n + 64,), MARK, device="cuda", dtype=dtype)
        v = full[16 + self.offset:16 + self.offset + n].view(shape)
        if values is not None:
            v.copy_(torch.from_numpy(values))
        self.made.append((full, v))
        return v

    def untouched(self):
        return all(bool((f[:v.storage_offset()] == MARK).all() and (f[v.storage_offset() + v.numel():] == MARK).all())
                   for f, v in self.made)


# rows of a wave and of several waves, at most 64 columns, longer than the
# registers hold; the fused backward (f16 with even N: four reserved rows where
# dx is 4-byte aligned, else five)
@pytest.mark.parametrize("M,N,dtype", [(7, 65, F32), (9, 33, F32), (5, 1000, F32), (4, 4099, F32), (3, 16385, F32),
                                       (2048, 2050, F32), (3584, 35, F32), (6, 61, F16), (6, 1000, F16),
                                       (4, 4099, F16), (3, 32769, F16), (3584, 34, F16), (3584, 67, F16),
                                       (2048, 4098, F16)])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_layernorm_at_any_address(C, M, N, dtype, offset):
    r, cv = rng(M + N), Canvas(offset)
    tol = 1e-5 if dtype == F32 else 2e-3
    x = cv.view((M, N), dtype, r.standard_normal((M, N)) * 2 + 0.5)
    g, b = cv.view((N,), dtype, r.standard_normal(N)), cv.view((N,), dtype, r.standard_normal(N))
    y, mean, rstd = cv.view((M, N), dtype), cv.view((M,), F32), cv.view((M,), F32)
    C.op_call(C.OpKind.LayerNormFwd, [x, g, b], [y, mean, rstd], LNEP, struct.pack("<f", 1e-5))
    y_ref, mu_ref, rs_ref = orc.layernorm_fwd_f64(host(x), host(g), host(b), eps=1e-5)
    assert orc.rel_err(host(y), y_ref) < tol
    assert orc.rel_err(host(mean), mu_ref) < 1e-5 and orc.rel_err(host(rstd), rs_ref) < 1e-5
    dy, dx = cv.view((M, N), dtype, r.standard_normal((M, N))), cv.view((M, N), dtype)
    dg, db = cv.view((N,), F32), cv.view((N,), F32)
    C.op_call(C.OpKind.LayerNormBwd, [x, dy, g, mean, rstd], [dx, dg, db])
    dx_ref, dg_ref, db_ref = orc.layernorm_bwd_f64(host(x), host(dy), host(mean), host(rstd), host(g))
    assert orc.rel_err(host(dx), dx_ref) < tol
    assert orc.rel_err(host(dg), dg_ref) < 1e-5 and orc.rel_err(host(db), db_ref) < 1e-5
    assert cv.untouched()


# a channel in registers; split over workgroups, in vectors of 8, 4 and 1
@pytest.mark.parametrize("shape", [(4, 5, 8, 8), (32, 6, 56, 56), (83, 3, 28, 28), (180, 2, 14, 14), (200, 3, 7, 7)])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_batchnorm_at_any_address(C, shape, offset):
    r, cv, Cc = rng(sum(shape)), Canvas(offset), shape[1]
    x = cv.view(shape, F16, r.standard_normal(shape) * 1.5 + 0.25)
    g, b = cv.view((Cc,), F16, r.standard_normal(Cc)), cv.view((Cc,), F16, r.standard_normal(Cc))
    y, mean, rstd = cv.view(shape, F16), cv.view((Cc,), F32), cv.view((Cc,), F32)
    C.op_call(C.OpKind.BatchNormFwd, [x, g, b], [y, mean, rstd], BNEP, struct.pack("<fI", 1e-5, 0))
    y_ref, mu_ref, rs_ref = orc.batchnorm_fwd_train_f64(host(x), host(g), host(b), eps=1e-5)
    assert orc.rel_err(host(y), y_ref) < 2e-3
    assert orc.rel_err(host(mean), mu_ref) < 1e-5 and orc.rel_err(host(rstd), rs_ref) < 1e-5
    dy, dx = cv.view(shape, F16, r.standard_normal(shape)), cv.view(shape, F16)
    dg, db = cv.view((Cc,), F32), cv.view((Cc,), F32)
    C.op_call(C.OpKind.BatchNormBwd, [x, dy, g, mean, rstd], [dx, dg, db])
    dx_ref, dg_ref, db_ref = orc.batchnorm_bwd_f64(host(x), host(dy), host(g), host(mean), host(rstd))
    assert orc.rel_err(host(dx), dx_ref) < 2e-3
    assert orc.rel_err(host(dg), dg_ref) < 1e-5 and orc.rel_err(host(db), db_ref) < 1e-5
    yi = cv.view(shape, F16)
    C.op_call(C.OpKind.BatchNormFwd, [x, g, b, mean, rstd], [yi], BNEP, struct.pack("<fI", 1e-5, 1))
    assert orc.rel_err(host(yi), orc.batchnorm_fwd_infer_f64(host(x), host(mean), host(rstd), host(g), host(b),
                                                             eps=1e-5)) < 2e-3
    assert cv.untouched()


def test_batchnorm_of_more_channels_than_a_grid_dimension(C):
    """65537 channels past the register limit: one workgroup each (their 8193
    elements are a channel of two values, whose mean and variance are known)."""
    N, Cc, H, W = 1, 65537, 3, 2731
    n = H * W
    lo, hi = (n + 1) // 2, n // 2  # how many of -1 and of +1
    x = torch.ones((N, Cc, H, W), device="cuda", dtype=F16)
    x.view(Cc, n)[:, ::2] = -1
    mu = (hi - lo) / n
    var = 1 - mu * mu
    y, mean, rstd = torch.zeros_like(x), torch.zeros(Cc, device="cuda"), torch.zeros(Cc, device="cuda")
    C.op_call(C.OpKind.BatchNormFwd, [x], [y, mean, rstd], BNEP, struct.pack("<fI", 1e-5, 0))
    assert float((mean - mu).abs().max()) < 1e-5 and float((rstd * (var + 1e-5) ** 0.5 - 1).abs().max()) < 1e-5
    for s in ((0, -1), (1, 1)):
        want = (s[1] - mu) / (var + 1e-5) ** 0.5
        assert float((y.view(Cc, n)[:, s[0]::2].float() - want).abs().max()) < 2e-3
    del y
    g = torch.ones(Cc, device="cuda", dtype=F16)
    dx, dg, db = torch.zeros_like(x), torch.zeros(Cc, device="cuda"), torch.zeros(Cc, device="cuda")
    C.op_call(C.OpKind.BatchNormBwd, [x, x, g, mean, rstd], [dx, dg, db])  # dy = x
    r = (var + 1e-5) ** -0.5
    assert float((db - (hi - lo)).abs().max()) < 1e-3  # whole numbers
    assert float((dg / (n * var * r) - 1).abs().max()) < 1e-4  # fp32 sums of 33 terms a lane
    for s in ((0, -1.0), (1, 1.0)):  # dx = r (dy - db / n - xhat dg / n) is r d eps / (var + eps)
        d = s[1] - mu
        assert float((dx.view(Cc, n)[:, s[0]::2].float() - r * (d - d * var * r * r)).abs().max()) < 1e-3
