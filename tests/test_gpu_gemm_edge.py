"""GPU parity of the GEMM at sizes and alignments that no tile divides: K that
ends inside a 16-byte chunk, a chunk and a K-step early or late, edge tiles of
one row or column, odd leading dimensions and odd base addresses, in all four
operand layouts and every epilogue; each of the kernel's tile and K-split
configurations; and shapes whose last exact tiles overlap their neighbours.
Operands and outputs are views into memory full of NaN: a
load that reads past an edge and counts, or a store outside the output, shows.

Tolerances (normwise against fp64 products of the stored operands): fp32
accumulation 1e-5 for fp32 outputs (K <= 1100), one output rounding for 16-bit
ones (bf16 2^-8, f16 2^-11, of the largest value).
"""
from __future__ import annotations

import struct

import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu

GEPI = int.from_bytes(b"GEPI", "little")
DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
TOL = {torch.float32: 1e-5, torch.float16: 2.0 ** -11 + 1e-5, torch.bfloat16: 2.0 ** -8 + 1e-5}


def view(values, ld_pad, offset, dtype, device="cuda"):
    """A [r, c] view of the values with row stride c + ld_pad, inside NaNs."""
    r, c = values.shape
    ld = c + ld_pad
    full = torch.full((r * ld + 2 * 64 + offset,), float("nan"), dtype=dtype, device=device)
    v = full[64 + offset:64 + offset + r * ld].view(r, ld)[:, :c]
    v.copy_(values)
    return full, v


def only_view_written(full, v):
    keep = torch.isnan(full)
    mask = torch.zeros_like(keep)
    torch.as_strided(mask, v.shape, v.stride(), v.storage_offset()).fill_(True)
    return bool((keep | mask).all()) and not bool(torch.isnan(v).any())


def gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def dgelu64(x):
    x = x.clone().requires_grad_(True)
    gelu64(x).sum().backward()
    return x.grad


# (M, N, K, pad of the leading dimensions, base offset in elements)
SIZES = [(1, 1, 8, 0, 0), (9, 3, 8, 1, 1), (64, 64, 9, 0, 0), (17, 10, 15, 3, 2), (65, 63, 63, 0, 0), (63, 65, 65, 1, 3),
         (129, 127, 64, 1, 0), (100, 72, 71, 0, 1), (8, 200, 127, 5, 0), (200, 8, 129, 0, 0),
         # K split 8 ways on 32 x 32, 4 ways on 64 x 32 and on 64 x 64 tiles
         (64, 10, 784, 0, 0), (33, 257, 1031, 1, 1), (500, 511, 523, 0, 0), (517, 700, 519, 1, 0),
         (650, 1000, 525, 0, 1), (1000, 1001, 1023, 0, 0),
         (192, 256, 4160, 0, 0), (512, 1024, 576, 0, 0),  # the same where the tiles divide the shape
         (1030, 1029, 72, 0, 0), (2049, 520, 40, 1, 1),  # 64 x 64 tiles, short K
         (2050, 1031, 40, 1, 1), (2048, 1024, 192, 0, 0),  # 64 x 128
         (2050, 1031, 265, 1, 1), (1100, 2051, 784, 0, 0),  # 128 x 64
         (2561, 2051, 255, 0, 0), (2600, 2500, 264, 8, 8),  # 128 x 128
         (3600, 3599, 520, 0, 0), (3333, 4099, 1000, 0, 1),  # 256 x 256
         # whole K-steps: the exact tiles, the last ones moved back (64, 128 and 256 wide, each pipeline depth)
         (250, 248, 128, 0, 0), (249, 248, 1024, 8, 8), (1530, 1400, 192, 0, 0), (1528, 1400, 1024, 0, 0),
         (2810, 3064, 128, 0, 0), (2808, 3064, 576, 8, 8), (4090, 4088, 128, 0, 0)]


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "bf16_f32"])
@pytest.mark.parametrize("size", SIZES)
def test_gemm_edges(C, size, dt):
    M, N, K, pad, offset = size
    din = DT[dt.split("_")[0]]
    dout = torch.float32 if "_" in dt else din
    cpad = 0 if dt == "f16" else pad  # the f16 variants take a contiguous output
    g = torch.Generator(device="cuda")
    g.manual_seed(M * 31 + N * 7 + K)
    a = torch.randn((M, K), device="cuda", generator=g).to(din)
    b = torch.randn((K, N), device="cuda", generator=g).div_(K ** 0.5).to(din)
    ref = a.double() @ b.double()
    bias = torch.randn(N, device="cuda", generator=g).to(din)
    z = torch.randn((M, N), device="cuda", generator=g).to(dout)
    for ta in (0, 1):
        for tb in (0, 1):
            _, A = view(a.T if ta else a, pad, offset, din)
            _, B = view(b.T if tb else b, pad, offset, din)
            full, out = view(torch.zeros((M, N), device="cuda"), cpad, offset, dout)
            out.fill_(float("nan"))
            C.op_call(C.OpKind.Gemm, [A, B], [out], 0, struct.pack("<ii", ta, tb))
            assert orc.rel_err(out.double().cpu().numpy(), ref.cpu().numpy()) < TOL[dout], (ta, tb)
            assert only_view_written(full, out)
            # epilogues: bias, bias + ReLU, bias + GELU (one layout each with the pre-activation), dGELU
            for kind in (1, 0, 3, 5):
                if dt == "bf16_f32" and kind != 1:
                    continue
                full, out = view(torch.zeros((M, N), device="cuda"), cpad, offset, dout)
                out.fill_(float("nan"))
                outs, x = [out], (bias.float() if "_" in dt else bias) if kind != 5 else z
                pre = ref + bias.double() if kind != 5 else ref
                if kind == 3 and ta == tb:
                    zfull, zout = view(torch.zeros((M, N), device="cuda"), pad, offset, dout)
                    zout.fill_(float("nan"))
                    outs.append(zout)
                C.op_call(C.OpKind.GemmEpilogue, [A, B, x], outs, GEPI, struct.pack("<iii", ta, tb, kind))
                want = {1: pre, 0: torch.relu(pre), 3: gelu64(pre), 5: ref * dgelu64(z.double())}[kind]
                assert orc.rel_err(out.double().cpu().numpy(), want.cpu().numpy()) < TOL[dout], (ta, tb, kind)
                assert only_view_written(full, out)
                if len(outs) == 2:
                    assert orc.rel_err(zout.double().cpu().numpy(), pre.cpu().numpy()) < TOL[dout]
                    assert only_view_written(zfull, zout)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
def test_gemm_nan_and_inf_stay_in_their_rows(C, dt):
    """A NaN or infinity in one row of A or one column of B reaches only its
    own row or column, at every distance from K's end."""
    M, N, K = 70, 69, 77
    a = torch.randn((M, K), device="cuda").to(DT[dt])
    b = torch.randn((K, N), device="cuda").to(DT[dt])
    a[3, 0] = float("nan")
    a[40, K - 1] = float("inf")
    b[0, 5] = float("inf")
    b[K - 1, 60] = float("nan")
    for ta in (0, 1):
        for tb in (0, 1):
            out = torch.empty((M, N), device="cuda", dtype=DT[dt])
            C.op_call(C.OpKind.Gemm, [a.T.contiguous() if ta else a, b.T.contiguous() if tb else b], [out], 0,
                      struct.pack("<ii", ta, tb))
            bad = ~torch.isfinite(out)
            want = torch.zeros_like(bad)
            want[[3, 40]] = True
            want[:, [5, 60]] = True
            assert torch.equal(bad, want)
