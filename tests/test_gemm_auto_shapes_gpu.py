"""The int8 GEMM (npu_kernels.py:40-56) on the tile the library picks by itself, over seeded random
ragged shapes that cross the picker's rules (M around 1024 and past 8192, K from one k-tile to
12288, N from one 16-column tile to the double-wide gate/up): int32 bit-exact against an fp64
product on the GPU (every product and partial sum is an integer below 2^53, so the fp64 result is
exact), the dequant epilogue bit-exact against bf16((acc.float() * sx) * sw) (pipeline.py:55-57) and
the residual epilogue against that plus the residual in bf16."""
import numpy as np
import pytest
import torch

from w8a8 import lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def shapes():
    rng = np.random.default_rng(2026)
    out = []
    for lo, hi in ((1, 300), (300, 1100), (1000, 1100), (1100, 4200), (4000, 4200), (8190, 8400)):
        for _ in range(3):
            M = int(rng.integers(lo, hi + 1))
            N = int(rng.integers(1, 820)) * 16
            K = int(rng.choice([64, 128, 1536, 2048, 6144, 12288, int(rng.integers(1, 100)) * 64]))
            out.append((M, N, K))
    out += [(3658, 24576, 1536), (3658, 1536, 12288), (512, 12288, 1536), (17, 16, 64)]
    return out


@pytest.mark.parametrize("M,N,K", shapes())
def test_auto_tile_int32_and_dequant_exact(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * 31 + N * 7 + K)
    a = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8, device=DEV)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8, device=DEV)
    sx = torch.rand(M, generator=g, device=DEV) * 0.05 + 1e-3
    sw = torch.rand(N, generator=g, device=DEV) * 0.015 + 0.005
    pw = ops.pack_weight(w, "nk", sw=sw)
    print(f"auto tile M={M} N={N} K={K}", flush=True)
    c = ops.gemm_i32(a, pw)
    want = (a.double() @ w.double().T).long()
    assert torch.equal(c.long(), want), f"int32 mismatch at M={M} N={N} K={K}"
    y = ops.gemm_bf16(a, sx, pw)
    ref = ((want.int().float() * sx[:, None]) * sw[None, :]).to(torch.bfloat16)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16)), f"dequant mismatch at M={M} N={N} K={K}"
    r = torch.randn(M, N, generator=g, device=DEV).to(torch.bfloat16)
    yr = ops.gemm_bf16(a, sx, pw, epilogue="residual", residual=r)
    assert torch.equal(yr.view(torch.int16), (ref + r).view(torch.int16)), f"residual mismatch at M={M} N={N} K={K}"


# Launches whose tiles of one size just fill the 256 CUs, and one tile more: 64x64, 64x128, and the
# BMx256 tiles (also at the share of the CUs the two largest must fill), short K, GELU pairs.
EDGES = [(64, 16384, 512), (64, 16400, 512), (4096, 256, 2048), (4097, 256, 2048), (128, 8208, 2048), (1024, 2048, 2048),
         (1025, 2048, 2048), (96, 16400, 512), (1536, 4096, 2048), (1537, 4096, 2048), (2100, 4096, 2048),
         (2560, 3600, 2048), (1280, 4400, 2048), (3072, 4096, 2048), (511, 2048, 448), (511, 2064, 448), (300, 24576, 512),
         (511, 8960, 1984), (512, 8960, 1984), (2100, 4096, 1984)]
# Fewer than 512 rows and K in [512, 2048) on each BMx256 tile, with the configuration that is meant: BM = 96,
# 128 (all 256 of its tiles, and a ragged last row tile), 160, 192 (with GELU 64x256 instead), and 64 past one round.
WIDE = {(150, 22016, 576): 7, (256, 32768, 512): 6, (250, 22080, 1040): 6, (385, 18688, 512): 8, (480, 21760, 1984): 8,
        (511, 18688, 960): 9, (500, 21760, 1536): 9, (500, 24576, 512): 4}


@pytest.mark.parametrize("M,N,K", EDGES + list(WIDE))
def test_auto_tile_exact_at_the_one_round_edges(M, N, K):
    cfg = lib().w8a8_gemm_pick_tile_config(M, N, K, 0)
    assert cfg == WIDE.get((M, N, K), cfg)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8, device=DEV)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8, device=DEV)
    sx, sw = torch.rand(M, generator=g, device=DEV) * 0.05, torch.rand(N, generator=g, device=DEV) * 0.01
    print(f"one-round edge M={M} N={N} K={K}", flush=True)
    want = (a.double() @ w.double().T).int()
    assert torch.equal(ops.gemm_i32(a, ops.pack_weight(w, "nk")), want)
    y = ((want.float() * sx[:, None]) * sw[None, :]).to(torch.bfloat16)
    assert torch.equal(ops.gemm_bf16(a, sx, ops.pack_weight(w, "nk", sw=sw)), y)
    if N % 64 == 0 and N <= 24576:  # what the row kernel of the reference result takes
        got = ops.gemm_bf16(a, sx, ops.pack_weight(w, "nk", N // 2, sw=sw), epilogue="gelu")
        assert torch.equal(got, ops.gelu_mul_bf16(y))
