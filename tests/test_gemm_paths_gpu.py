"""GPU parity of paths that the default dispatch takes for other products than the small ones of
test_gemm_chain_gpu.py: the wave tiles with all their leaves on (config bit 0x40000 keeps a product on
them), launches of more than 256 workgroups on the 16-row tiles, and the f32 MFMA against the fmaf chain
where no rounding follows the sum."""
import numpy as np
import pytest
import torch

import oracle
from conftest import assert_bits
from test_gemm_chain_gpu import HALF, HALF_EXT, HALF_WIDE, _accums, _operands, _run

pytestmark = pytest.mark.gpu

WAVE = 0x40000


@pytest.mark.parametrize("values", ["uniform", "e4m3", "wide", "tiny", "large", "special"])
@pytest.mark.parametrize("kind", [1, 7, 10, 20, 23, HALF, HALF_EXT, HALF_WIDE], ids=str)
def test_wave_tiles(dev, kind, values):
    import lofloat_amd as lof
    M, N, K = 66, 130, 131
    A, B = _operands(M, N, K, values, seed=12)
    for chunk in (1, 2, 4, 8, 16, 32):
        acc, oacc = _accums(lof, kind, chunk)
        ref = oracle.gemm(A, B, oacc, alpha=0.75)
        for cfg in range(5, 9):
            got = _run(lof, A, B, acc, dev, cfg % 2 == 0, True, cfg | WAVE, False)
            assert_bits(got, ref, f"{kind} {values} chunk {chunk} config {cfg}")


@pytest.mark.parametrize("bits", [10, 23, HALF], ids=str)
def test_wave_tile_leaf_changes(dev, bits):
    """Chunk 1 from exact and held leaves to directed and general ones and back, within one product."""
    import lofloat_amd as lof
    M, N, K = 70, 66, 520
    g = np.random.default_rng(32)
    A, B = (oracle.virtual_round(g.standard_normal(s).astype(np.float32).ravel(),
                                 (8, 3, 7, 1, 0, 0)).reshape(s) for s in ((M, K), (K, N)))
    A[:, 200:230] = g.standard_normal((M, 30))
    A[:, 300:340] = 0.0
    B[360:400] *= np.float32(2.0 ** 40)
    A[5, 450] = np.float32(1 + 2.0 ** -23)
    acc, oacc = _accums(lof, bits, 1)
    ref = oracle.gemm(A, B, oacc, alpha=0.75)
    for cfg in range(5, 9):
        assert_bits(_run(lof, A, B, acc, dev, 0, 1, cfg | WAVE, False), ref, f"config {cfg}")


@pytest.mark.parametrize("chunk", [1, 8, 32])
def test_wave_tile_conv(dev, chunk):
    import lofloat_amd as lof
    g = np.random.default_rng(6)
    x = g.uniform(-1, 1, (2, 5, 13, 13)).astype(np.float32)
    w = g.uniform(-1, 1, (70, 5, 3, 3)).astype(np.float32)
    for kind in (10, 23, HALF):
        acc, oacc = _accums(lof, kind, chunk)
        ref = oracle.conv2d(x, w, oacc, pad=(1, 1), stride=(1, 1))
        for cfg in (6, 7):
            y = lof.conv2d(torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), acc, padding=1,
                           config=cfg | WAVE).cpu().numpy()
            assert_bits(y, ref, f"{kind} chunk {chunk} config {cfg}")


@pytest.mark.parametrize("kind", [7, 10, 23])
@pytest.mark.parametrize("K", [7, 70])
def test_more_than_256_workgroups_of_16_rows(dev, kind, K):
    """Chunk 1 on FP32 operands: launches past 256 workgroups switch the rounding mode in every leaf, up
    to 256 they stay in round-down."""
    import lofloat_amd as lof
    M, N = 601, 533      # 323 tiles of 32x32, 342 of 16x64, 340 of 64x16, 1292 of 16x16
    A, B = _operands(M, N, K, "uniform", seed=K)
    acc, oacc = _accums(lof, kind, 1)
    ref = oracle.gemm(A, B, oacc, alpha=0.75)
    for cfg in (9, 10, 11, 12):
        for ta, tb in ((0, 1), (1, 0)):
            assert_bits(_run(lof, A, B, acc, dev, ta, tb, cfg, False), ref, f"{kind} config {cfg}")


@pytest.mark.parametrize("chunk", [4, 8, 32])
@pytest.mark.parametrize("scale", [0, 20, 60, 110, -60, -75])
def test_mfma_is_the_fmaf_chain_unrounded(dev, scale, chunk):
    """Sums into 23-bit accumulators, which keep every float, over several chunks."""
    import lofloat_amd as lof
    g = torch.Generator(device=dev).manual_seed(scale + 100 + chunk)
    acc = lof.AccumSpec(mant_bits=23, chunk=chunk)
    spread = abs(scale) if scale < 100 else 12
    A, B = ((torch.rand(1024, 3 * chunk, device=dev, generator=g) * 2 - 1) *
            torch.exp2(torch.randint(-spread, 1, (1024, 3 * chunk), device=dev, generator=g) / 2 + scale / 2)
            for _ in range(2))
    ref = lof.gemm(A, B.t(), acc, config=7 | 0x200)
    for cfg in (5, 7, 9, 10, 11):
        got = lof.gemm(A, B.t(), acc, config=cfg)
        same = (got.view(torch.int32) == ref.view(torch.int32)) | (got.isnan() & ref.isnan())
        assert bool(same.all()), (scale, chunk, cfg, int((~same).sum()))
