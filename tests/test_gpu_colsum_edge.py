"""GPU parity of the one-output column sum at widths that are no multiple of a
16-byte vector, at odd base addresses, and around the switch to 1024 threads
(M = 256, 128 column blocks), f32, f16 and bf16 in, against fp64: 1e-5 for
fp32 outputs (sums of at most 4100 values), one rounding for f16 ones."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "f16_f16"])
@pytest.mark.parametrize("M,N", [(1, 4), (3, 8), (5, 9), (777, 523), (256, 17), (257, 17), (4100, 10), (4099, 31),
                                 (2048, 1024), (300, 1025), (300, 2049), (1000, 3), (513, 4099)])
@pytest.mark.parametrize("offset", [0, 1])
def test_column_sum_edges(C, M, N, dt, offset):
    din = DT[dt.split("_")[0]]
    dout = torch.float16 if "_" in dt else torch.float32
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    full = torch.full((M * N + 64,), float("nan"), device="cuda", dtype=din)
    x = full[16 + offset:16 + offset + M * N].view(M, N)
    x.copy_(torch.randn((M, N), device="cuda", generator=g) + 0.25)
    of = torch.full((N + 64,), 77.0, device="cuda", dtype=dout)
    o = of[16:16 + N]
    C.op_call(C.OpKind.ReduceSum, [x], [o])
    ref = x.double().sum(0)
    tol = 1e-5 if dout == torch.float32 else 2.0 ** -11 + 1e-5
    assert float((o.double() - ref).abs().max() / ref.abs().max()) < tol
    assert bool((of[:16] == 77).all()) and bool((of[16 + N:] == 77).all())


@pytest.mark.parametrize("dt,M,N", [("f32", 777, 523), ("f32", 300, 9), ("f32", 500, 1001), ("f32", 300, 1024),
                                    ("f16", 777, 517), ("f16", 300, 17), ("f16", 500, 1024)])
@pytest.mark.parametrize("row", [0, -1])
def test_column_sum_over_a_row_of_its_input(C, dt, M, N, row):
    """The sums may take the place of a row: a workgroup has read its columns
    when it writes them, and no other one reads them."""
    g = torch.Generator(device="cuda")
    g.manual_seed(M * N)
    x = (torch.randn((M, N), device="cuda", generator=g) + 0.25).to(DT[dt])
    ref = x.double().sum(0)
    C.op_call(C.OpKind.ReduceSum, [x], [x[row]])
    tol = 1e-5 if dt == "f32" else 2.0 ** -11 + 1e-5
    assert float((x[row].double() - ref).abs().max() / ref.abs().max()) < tol


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("M,N", [(191, 33), (192, 33), (1023, 3100), (1024, 3100), (1023, 6200), (1024, 6200),
                                 (192, 12300), (1030, 12300), (4096, 16), (4097, 8), (4095, 16)])
def test_column_sum_around_its_rules(C, M, N, dt):
    """The widths and row counts at which the kernel changes."""
    for offset in (0, 1):
        test_column_sum_edges(C, M, N, dt, offset)
