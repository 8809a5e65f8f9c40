"""The GEMM epilogues with AdamW and with column partials on the tiles that
small matrices take (64 x 64 and 128 x 128, each pipeline depth) as well as
on 256 x 256: bit-identical to the separate ops (fp32-output GEMM, then
adamw_step; dGELU GEMM), the partials against fp64 sums of the stored output
(256 values each, 1e-5 normwise)."""
from __future__ import annotations

import struct

import pytest
import torch

pytestmark = pytest.mark.gpu

GADW, ADAM, GEPI = (int.from_bytes(t, "little") for t in (b"GADW", b"ADAM", b"GEPI"))
HYPER = (1e-3, 0.9, 0.999, 1e-8, 0.01)


@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (256, 512, 1024), (512, 768, 192), (1536, 1536, 192),
                                   (1536, 1536, 1088), (2048, 2560, 1024), (4096, 2048, 128)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_adamw_tiles(C, M, N, K, ta, tb):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    a = torch.randn((K, M) if ta else (M, K), device="cuda", generator=g).bfloat16()
    b = torch.randn((N, K) if tb else (K, N), device="cuda", generator=g).bfloat16()
    P = torch.randn((M, N), device="cuda", generator=g)
    m, v = torch.randn((M, N), device="cuda", generator=g), torch.rand((M, N), device="cuda", generator=g)
    step = torch.full((), 3, device="cuda", dtype=torch.int32)
    ref = [t.clone() for t in (P, m, v)] + [P.bfloat16()]
    got = [t.clone() for t in (P, m, v)] + [P.bfloat16()]
    G = torch.empty((M, N), device="cuda")
    C.launch_by_id("gemm_bf16_mfma_f32out_v0", C.OpKind.Gemm, [a, b], [G], 0, struct.pack("<ii", ta, tb))
    C.launch_by_id("adamw_step_f32_v1", C.OpKind.AdamStep, ref[:1] + [G] + ref[1:3] + [step], ref, ADAM,
                   struct.pack("<fffff", *HYPER))
    C.launch_by_id("gemm_adamw_bf16_v0", C.OpKind.GemmAdamW, [a, b] + got[:3] + [step], got, GADW,
                   struct.pack("<iifffff", ta, tb, *HYPER))
    for x, y in zip(got, ref):
        assert torch.equal(x, y)


@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (256, 3584, 512), (512, 768, 1024), (1536, 1536, 192),
                                   (2048, 2048, 1024), (2816, 3072, 128)])
@pytest.mark.parametrize("tb", [0, 1])
def test_dgelu_column_partials_tiles(C, M, N, K, tb):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    a = torch.randn((M, K), device="cuda", generator=g).bfloat16()
    b = torch.randn((N, K) if tb else (K, N), device="cuda", generator=g).mul_(K ** -0.5).bfloat16()
    z = torch.randn((M, N), device="cuda", generator=g).bfloat16()
    plain, out = (torch.empty((M, N), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    part = torch.full((M // 256, N), float("nan"), device="cuda")
    C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [plain], GEPI, struct.pack("<iii", 0, tb, 5))
    C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [out, part], GEPI, struct.pack("<iii", 0, tb, 7))
    assert torch.equal(out, plain)
    ref = out.double().view(M // 256, 256, N).sum(1)
    assert float((part.double() - ref).abs().max() / ref.abs().max()) < 1e-5
    db, ws = torch.empty(N, device="cuda"), torch.empty((M // 256, N), device="cuda")
    C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [out, db, ws], GEPI, struct.pack("<iii", 0, tb, 6))
    assert torch.equal(ws, part)
    assert float((db.double() - ref.sum(0)).abs().max() / ref.sum(0).abs().max()) < 1e-5


@pytest.mark.parametrize("M,N", [(300, 256), (512, 264), (500, 520)])
def test_ragged_shapes_stay_refused(C, M, N):
    """Shapes that a plain GEMM runs on tiles moved back are no shapes for
    column sums or an update in place."""
    a, b = torch.zeros((M, 64), device="cuda").bfloat16(), torch.zeros((64, N), device="cuda").bfloat16()
    z, out = (torch.zeros((M, N), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    part = torch.empty((M // 256, N), device="cuda")
    with pytest.raises(RuntimeError, match="NotImplemented"):
        C.op_call(C.OpKind.GemmEpilogue, [a, b, z], [out, part], GEPI, struct.pack("<iii", 0, 0, 7))
    with pytest.raises(RuntimeError, match="InvalidArgument"):
        C.launch_by_id("gemm_epilogue_bf16_mfma_v0", C.OpKind.GemmEpilogue, [a, b, z], [out, part], GEPI,
                       struct.pack("<iii", 0, 0, 7))
    P, m, v = (torch.zeros((M, N), device="cuda") for _ in range(3))
    step = torch.ones((), device="cuda", dtype=torch.int32)
    with pytest.raises(RuntimeError, match="InvalidArgument"):
        C.launch_by_id("gemm_adamw_bf16_v0", C.OpKind.GemmAdamW, [a, b, P, m, v, step], [P, m, v, P.bfloat16()], GADW,
                       struct.pack("<iifffff", 0, 0, *HYPER))


@pytest.mark.parametrize("M,N,K", [(256, 256, 1984), (256, 256, 2048), (256, 1024, 2048), (512, 512, 4032),
                                   (512, 512, 4096), (1024, 256, 4096), (512, 768, 4096)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_adamw_of_long_k(C, M, N, K, ta, tb):
    """Where the plain product splits K the fused one does too: same bits."""
    test_gemm_adamw_tiles(C, M, N, K, ta, tb)


@pytest.mark.parametrize("M,N,K", [(256, 1024, 2048), (256, 1024, 4096), (512, 512, 4096), (768, 512, 2048)])
@pytest.mark.parametrize("tb", [0, 1])
def test_dgelu_column_partials_of_long_k(C, M, N, K, tb):
    """The sums of a product that runs on the K-split tiles."""
    test_dgelu_column_partials_tiles(C, M, N, K, tb)
