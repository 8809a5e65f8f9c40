"""GPU parity of LayerNorm and BatchNorm at the sizes where their kernels
change: rows of one vector, rows that end inside a vector, the widest row of
each lane count, the fused affine backward (its smallest matrix, rows that do
not divide over its chunks, odd f16 rows), channels at the register limit and
just past it, and outputs that are an input's own memory.  Oracle and
tolerances as in test_gpu_norm.py: fp64 on the stored inputs, fp32 <= 1e-5,
f16 <= 2e-3 (one f16 rounding).
"""
from __future__ import annotations

import struct

import pytest
import torch

import oracle as orc
from test_gpu_norm import BNEP, LNEP, dev, host, rng

pytestmark = pytest.mark.gpu

F32, F16 = torch.float32, torch.float16
LN = [(1, 4, F32), (3, 5, F32), (2, 7, F32), (1, 8, F16), (3, 9, F16), (5, 15, F16), (9, 255, F32), (4, 257, F32),
      (7, 513, F16), (6, 1000, F16), (5, 1024, F32), (4, 1025, F32), (3, 2049, F32), (3, 4096, F32), (2, 4099, F16),
      (3, 8191, F32), (2, 8193, F16), (2, 16384, F32), (2, 16385, F32), (1, 32768, F16), (300, 1000, F32),
      (1500, 264, F16),
      # the fused backward: 2048 rows, 16 MiB
      (2048, 2048, F32), (3583, 24, F32), (3584, 9, F16), (5000, 33, F32), (2303, 2050, F32), (4097, 1025, F32), (2048, 8192, F32), (4300, 2049, F16),
      (2056, 4098, F16), (2049, 8200, F16), (16390, 516, F16)]


@pytest.mark.parametrize("M,N,dtype", LN)
@pytest.mark.parametrize("affine", [False, True])
def test_layernorm_paths(C, M, N, dtype, affine):
    r = rng(M * 7 + N)
    tol = 1e-5 if dtype == F32 else 2e-3
    x = dev(r.standard_normal((M, N)) * 2 + 0.5, dtype)
    g, b = (dev(r.standard_normal(N), dtype), dev(r.standard_normal(N), dtype)) if affine else (None, None)
    y, mean, rstd = torch.empty_like(x), torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    C.op_call(C.OpKind.LayerNormFwd, [x, g, b] if affine else [x], [y, mean, rstd], LNEP, struct.pack("<f", 1e-5))
    xs, (gs, bs) = host(x), (host(g), host(b)) if affine else (None, None)
    y_ref, mu_ref, rs_ref = orc.layernorm_fwd_f64(xs, gs, bs, eps=1e-5)
    assert orc.rel_err(host(mean), mu_ref) < 1e-5 and orc.rel_err(host(rstd), rs_ref) < 1e-5
    assert orc.rel_err(host(y), y_ref) < tol
    dy = dev(r.standard_normal((M, N)), dtype)
    dx, dg, db = torch.empty_like(x), torch.empty(N, device="cuda"), torch.empty(N, device="cuda")
    ref = orc.layernorm_bwd_f64(xs, host(dy), host(mean), host(rstd), gs)
    ins = [x, dy, g, mean, rstd] if affine else [x, dy, mean, rstd]
    C.op_call(C.OpKind.LayerNormBwd, ins, [dx, dg, db] if affine else [dx])
    for got, want, t in ((dx, ref[0], tol),) + (((dg, ref[1], 1e-5), (db, ref[2], 1e-5)) if affine else ()):
        assert orc.rel_err(host(got), want) < t
    # in place: dx is dy, then x (the sums are taken before it is overwritten)
    for k in (1, 0):
        own = [t.clone() for t in (x, dy)]
        C.op_call(C.OpKind.LayerNormBwd, own + ins[2:], [own[k], dg, db] if affine else [own[k]])
        assert orc.rel_err(host(own[k]), ref[0]) < tol
        if affine:
            assert orc.rel_err(host(dg), ref[1]) < 1e-5 and orc.rel_err(host(db), ref[2]) < 1e-5
    C.op_call(C.OpKind.LayerNormFwd, [x, g, b] if affine else [x], [x, mean, rstd], LNEP, struct.pack("<f", 1e-5))
    assert torch.equal(x, y)


BN = [(1, 1, 1, 3), (2, 3, 7, 7), (10, 2, 7, 7), (128, 5, 7, 7), (11, 4, 5, 149), (200, 3, 7, 7), (4, 70, 2, 2),
      (5, 3, 14, 14), (21, 2, 14, 14), (83, 2, 14, 14), (167, 2, 14, 14), (180, 3, 14, 14), (8, 3, 16, 16),
      (83, 2, 28, 28), (84, 3, 28, 28), (9, 5, 128, 128), (3, 2, 1, 65536)]


@pytest.mark.parametrize("shape", BN)
@pytest.mark.parametrize("in_place", [False, True])
def test_batchnorm_paths(C, shape, in_place):
    r = rng(sum(shape))
    Cc = shape[1]
    x = dev(r.standard_normal(shape) * 1.5 + 0.25, F16)
    g, b = dev(r.standard_normal(Cc), F16), dev(r.standard_normal(Cc), F16)
    dy = dev(r.standard_normal(shape), F16)
    y_ref, mu_ref, rs_ref = orc.batchnorm_fwd_train_f64(host(x), host(g), host(b), eps=1e-5)
    xi = x.clone()
    y = xi if in_place else torch.empty_like(x)
    mean, rstd, dg, db = (torch.empty(Cc, device="cuda") for _ in range(4))
    C.op_call(C.OpKind.BatchNormFwd, [xi, g, b], [y, mean, rstd], BNEP, struct.pack("<fI", 1e-5, 0))
    assert orc.rel_err(host(mean), mu_ref) < 1e-5 and orc.rel_err(host(rstd), rs_ref) < 1e-5
    assert orc.rel_err(host(y), y_ref) < 2e-3
    dx_ref, dg_ref, db_ref = orc.batchnorm_bwd_f64(host(x), host(dy), host(g), host(mean), host(rstd))
    d = dy.clone()
    dx = d if in_place else torch.empty_like(x)
    C.op_call(C.OpKind.BatchNormBwd, [x, d, g, mean, rstd], [dx, dg, db])
    assert orc.rel_err(host(dx), dx_ref) < 2e-3
    assert orc.rel_err(host(dg), dg_ref) < 1e-5 and orc.rel_err(host(db), db_ref) < 1e-5
    rv = torch.rand(Cc, device="cuda") + 0.5
    yi = torch.empty_like(x)
    C.op_call(C.OpKind.BatchNormFwd, [x, g, b, mean, rv], [yi], BNEP, struct.pack("<fI", 1e-5, 1))
    ref = orc.batchnorm_fwd_infer_f64(host(x), host(mean), host(rv), host(g), host(b), eps=1e-5)
    assert orc.rel_err(host(yi), ref) < 2e-3
