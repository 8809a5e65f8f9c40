"""GPU parity of the GEMM on both sides of the rules that choose its tiles, in
all four operand layouts; against fp64 products of the stored operands, with
the tolerances of test_gpu_gemm_edge.py (K <= 1100: fp32 1e-5, 16-bit one
output rounding)."""
from __future__ import annotations

import struct

import pytest
import torch

import oracle as orc
from test_gpu_gemm_edge import DT, GEPI, TOL, dgelu64, gelu64

pytestmark = pytest.mark.gpu


def check(C, M, N, K, dt, kinds=()):
    din = DT[dt.split("_")[0]]
    dout = torch.float32 if "_" in dt else din
    g = torch.Generator(device="cuda")
    g.manual_seed(M * 31 + N * 7 + K)
    a = torch.randn((M, K), device="cuda", generator=g).to(din)
    b = torch.randn((K, N), device="cuda", generator=g).div_(K ** 0.5).to(din)
    bias, z = torch.randn(N, device="cuda", generator=g).to(dout), torch.randn((M, N), device="cuda", generator=g).to(dout)
    ref = a.double() @ b.double()
    for ta in (0, 1):
        for tb in (0, 1):
            A, B = a.T.contiguous() if ta else a, b.T.contiguous() if tb else b
            out = torch.full((M, N), float("nan"), device="cuda", dtype=dout)
            C.op_call(C.OpKind.Gemm, [A, B], [out], 0, struct.pack("<ii", ta, tb))
            assert orc.rel_err(out.double().cpu().numpy(), ref.cpu().numpy()) < TOL[dout], (ta, tb)
            for kind in kinds:
                out.fill_(float("nan"))
                outs = [out] + ([torch.empty_like(out)] if kind == 3 else [])
                C.op_call(C.OpKind.GemmEpilogue, [A, B, z if kind == 5 else bias], outs, GEPI,
                          struct.pack("<iii", ta, tb, kind))
                want = ref * dgelu64(z.double()) if kind == 5 else gelu64(ref + bias.double())
                assert orc.rel_err(out.double().cpu().numpy(), want.cpu().numpy()) < TOL[dout], (ta, tb, kind)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "bf16_f32"])
@pytest.mark.parametrize("M,N,K", [(1600, 1600, 704), (1600, 1600, 1024), (2048, 2112, 704), (2048, 2112, 768),
                                   (2944, 2944, 704), (2944, 2944, 1024), (4224, 4224, 768)])
def test_shapes_of_whole_smaller_tiles(C, M, N, K, dt):
    """Multiples of 64 and of 128 that larger tiles would have to move back."""
    check(C, M, N, K, dt, (3, 5) if dt != "bf16_f32" else ())


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("K", [448, 512])
def test_many_tiles_of_whole_64s(C, K, dt):
    check(C, 5824, 5696, K, dt)


@pytest.mark.parametrize("M,N,K", [(2048, 1536, 1024), (2048, 1792, 512), (2048, 1792, 544), (2048, 2048, 512),
                                   (2048, 2048, 1056), (2048, 2176, 1024), (3072, 2048, 128)])
def test_fp32_tiles_by_the_fullest_cu(C, M, N, K):
    check(C, M, N, K, "f32")


@pytest.mark.parametrize("M,N,K", [(512, 512, 508), (512, 512, 512), (1024, 256, 256), (528, 512, 320), (1000, 200, 319),
                                   (1000, 200, 320), (688, 512, 256), (704, 512, 256), (8000, 32, 320)])
def test_fp32_few_tiles(C, M, N, K):
    check(C, M, N, K, "f32")
