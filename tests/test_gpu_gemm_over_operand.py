"""GPU parity of products written over one of their operands, where one tile
spans the output's other dimension; against fp64 products of the operands as
they were (tolerances of test_gpu_gemm_edge.py)."""
from __future__ import annotations

import struct

import pytest
import torch

pytestmark = pytest.mark.gpu

GADW, ADAM, GEPI = (int.from_bytes(t, "little") for t in (b"GADW", b"ADAM", b"GEPI"))
HYPER = (1e-3, 0.9, 0.999, 1e-8, 0.01)
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
TOL = {"f32": 1e-5, "f16": 2.0 ** -11 + 1e-5, "bf16": 2.0 ** -8 + 1e-5}


def operands(M, N, K, dt):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    a = torch.randn((M, K), device="cuda", generator=g).to(DT[dt])
    return a, torch.randn((K, N), device="cuda", generator=g).mul_(K ** -0.5).to(DT[dt])


def err(got, want):
    return float((got.double() - want).abs().max() / want.abs().max())


# C in A's first N columns: exact 128 and 64 wide tiles, ragged M, K that a
# split would share out, sizes that no tile divides
@pytest.mark.parametrize("M,N,K,dt", [(16384, 128, 128, "f32"), (8192, 64, 512, "f32"), (8200, 48, 513, "f32"),
                                      (1000, 64, 64, "bf16"), (1000, 64, 64, "f16"), (64, 64, 4096, "bf16"),
                                      (40, 50, 2100, "bf16"), (300, 50, 50, "bf16"), (33024, 128, 128, "bf16")])
def test_product_over_a(C, M, N, K, dt):
    a, b = operands(M, N, K, dt)
    if dt == "f16":  # its output is contiguous
        assert N == K
    ref = a.double() @ b.double()
    C.op_call(C.OpKind.Gemm, [a, b], [a[:, :N]], 0, struct.pack("<ii", 0, 0))
    assert err(a[:, :N], ref) < TOL[dt]


@pytest.mark.parametrize("M,N,K,dt", [(64, 16384, 64, "f32"), (64, 1000, 64, "bf16"), (64, 64, 4096, "bf16")])
def test_product_over_b(C, M, N, K, dt):
    a, b = operands(M, N, K, dt)
    ref = a.double() @ b.double()
    C.op_call(C.OpKind.Gemm, [a, b], [b[:M]], 0, struct.pack("<ii", 0, 0))
    assert err(b[:M], ref) < TOL[dt]


def test_fused_epilogues_over_a(C):
    """One 256 x 256 tile: dGELU with column partials, and AdamW's shadow."""
    a, b = operands(256, 256, 256, "bf16")
    z = torch.randn((256, 256), device="cuda").bfloat16()
    want, wp, part = torch.empty_like(z), torch.empty((1, 256), device="cuda"), torch.empty((1, 256), device="cuda")
    C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [want, wp], GEPI, struct.pack("<iii", 0, 0, 7))
    own = a.clone()
    C.op_call(C.OpKind.GemmEpilogue, [own, b, z], [own, part], GEPI, struct.pack("<iii", 0, 0, 7))
    assert torch.equal(own, want) and torch.equal(part, wp)
    P, m, v = (torch.rand((256, 256), device="cuda") for _ in range(3))
    step = torch.ones((), device="cuda", dtype=torch.int32)
    runs = []
    for w in (torch.empty_like(a), a):
        s = [t.clone() for t in (P, m, v)]
        C.op_call(C.OpKind.GemmAdamW, [a, b] + s + [step], s + [w], GADW, struct.pack("<iifffff", 0, 0, *HYPER))
        runs.append(s + [w])
    for x, y in zip(*runs):
        assert torch.equal(x, y)


@pytest.mark.parametrize("M,N,K,dt", [(1000, 1000, 1024, "bf16"), (250, 248, 128, "f32"), (2808, 3064, 576, "f16"),
                                      (129, 127, 64, "bf16"), (517, 700, 519, "f32"), (2561, 2051, 255, "f16")])
def test_dgelu_over_its_own_pre_activation(C, M, N, K, dt):
    """At ragged shapes, on tiles moved back or not: each element of Z is read
    where the output's is stored."""
    a, b = operands(M, N, K, dt)
    z = torch.randn((M, N), device="cuda").to(DT[dt])
    apart = torch.empty_like(z)
    z64 = z.double().requires_grad_(True)
    torch.nn.functional.gelu(z64, approximate="tanh").sum().backward()
    ref = (a.double() @ b.double()) * z64.grad
    C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [apart], GEPI, struct.pack("<iii", 0, 0, 5))
    C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [z], GEPI, struct.pack("<iii", 0, 0, 5))
    assert err(z, ref) < TOL[dt] and err(apart, ref) < TOL[dt]
