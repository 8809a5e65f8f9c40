"""GPU parity of the normalisations where their sums are written over memory
that the same call reads (gamma, the saved statistics, the input), for every
form of the call; against the fp64 oracle on the inputs as they were,
with test_gpu_norm.py's tolerances (fp32 1e-5, f16 2e-3)."""
from __future__ import annotations

import pytest
import torch

import oracle as orc
from test_gpu_norm import dev, host, rng

pytestmark = pytest.mark.gpu

F32, F16 = torch.float32, torch.float16


def ln_inputs(M, N, dtype):
    r = rng(M * 5 + N)
    x, dy = dev(r.standard_normal((M, N)) * 2 + 0.5, dtype), dev(r.standard_normal((M, N)), dtype)
    x64 = host(x)
    mean, rstd = dev(x64.mean(1), F32), dev(1 / (x64.var(1) + 1e-5) ** 0.5, F32)
    return x, dy, dev(r.standard_normal(N), dtype), mean, rstd


def check_ln(ins, outs):
    (dx, dg, db), tol = outs, 1e-5 if ins[0].dtype == F32 else 2e-3
    return lambda ref: (orc.rel_err(host(dx), ref[0]) < tol and orc.rel_err(host(dg), ref[1]) < 1e-5
                        and orc.rel_err(host(db), ref[2]) < 1e-5)


# one launch; row by row in one and several waves; the fused form; rows wider
# than its columns; rows shorter than a vector and longer than the registers hold
@pytest.mark.parametrize("M,N,dtype", [(300, 1000, F32), (5, 24, F16), (40, 4099, F32), (2048, 2048, F32),
                                       (3584, 40, F32), (3584, 33, F16), (2048, 4100, F16), (5, 16384, F32),
                                       (6, 3, F32), (7, 5, F16), (3, 20001, F32)])
@pytest.mark.parametrize("which", ["dgamma", "dbeta"])
def test_layernorm_sums_over_gamma(C, M, N, dtype, which):
    x, dy, g, mean, rstd = ln_inputs(M, N, dtype)
    ref = orc.layernorm_bwd_f64(host(x), host(dy), host(mean), host(rstd), host(g))
    own = torch.zeros(N, device="cuda")
    gamma = own.view(dtype)[:N]
    gamma.copy_(g)
    dx, other = torch.empty_like(x), torch.empty(N, device="cuda")
    outs = [dx, own, other] if which == "dgamma" else [dx, other, own]
    C.op_call(C.OpKind.LayerNormBwd, [x, dy, gamma, mean, rstd], outs)
    assert check_ln([x], outs)(ref)


@pytest.mark.parametrize("n", [3, 8, 33, 64])
@pytest.mark.parametrize("onto", ["statistics", "rows"])
def test_layernorm_sums_over_what_one_workgroup_reads(C, n, onto):
    """Up to 64 columns: one workgroup has read every row when it writes."""
    x, dy, g, mean, rstd = ln_inputs(n, n, F32)
    ref = orc.layernorm_bwd_f64(host(x), host(dy), host(mean), host(rstd), host(g))
    outs = [torch.empty_like(x)] + ([mean, rstd] if onto == "statistics" else [x[0], dy[n - 1]])
    C.op_call(C.OpKind.LayerNormBwd, [x, dy, g, mean, rstd], outs)
    assert check_ln([x], outs)(ref)


# a channel in registers; split over workgroups, in vectors of 8, 4 and 1
BN = [(4, 5, 8, 8), (32, 6, 56, 56), (83, 3, 28, 28), (180, 2, 14, 14), (200, 3, 7, 7)]


@pytest.mark.parametrize("shape", BN)
@pytest.mark.parametrize("dx_on", [None, "x", "dy"])
def test_batchnorm_sums_over_the_saved_statistics(C, shape, dx_on):
    r = rng(sum(shape))
    Cc = shape[1]
    x, dy = dev(r.standard_normal(shape) * 1.5 + 0.25, F16), dev(r.standard_normal(shape), F16)
    g = dev(r.standard_normal(Cc), F16)
    x64 = host(x)
    mean, rstd = dev(x64.mean((0, 2, 3)), F32), dev(1 / (x64.var((0, 2, 3)) + 1e-5) ** 0.5, F32)
    ref = orc.batchnorm_bwd_f64(x64, host(dy), host(g), host(mean), host(rstd))
    dx = {None: torch.empty_like(x), "x": x, "dy": dy}[dx_on]
    C.op_call(C.OpKind.BatchNormBwd, [x, dy, g, mean, rstd], [dx, mean, rstd])
    assert orc.rel_err(host(dx), ref[0]) < 2e-3
    assert orc.rel_err(host(mean), ref[1]) < 1e-5 and orc.rel_err(host(rstd), ref[2]) < 1e-5
