"""GPU parity of the chunk-sum kernels (chunks 2 to 32, every chunk sum an f32 MFMA chain) and of
their chunk-1 form (directed, binary16-held and exact-sum leaves): every tile, at the edges of
tiles and slices, in all operand layouts and with odd leading dimensions, against the oracle bit
for bit; and the f32 MFMA against the VALU fmaf chain."""
import numpy as np
import pytest
import torch

import oracle
from conftest import assert_bits

pytestmark = pytest.mark.gpu

HALF, HALF_EXT, HALF_WIDE = (16, 10, 15, 1, 0, 0), (16, 10, 15, 0, 0, 0), (18, 10, 15, 1, 0, 0)
CONFIGS = range(5, 13)   # 128x128, 128x64, 64x64, 64x128, 32x32, 16x64, 64x16, 16x16


def _accums(lof, kind, chunk):
    if isinstance(kind, int):
        return lof.AccumSpec(mant_bits=kind, chunk=chunk), oracle.accum_mant(kind, chunk)
    fmt = lof.FloatFormatDescriptor(*kind, lof.formats.P3109_InfChecker(kind[0]),
                                    lof.formats.P3109_NaNChecker(kind[0]))
    return lof.AccumSpec(fmt=fmt, chunk=chunk), oracle.accum_fmt(kind, chunk)


def _operands(M, N, K, values, seed):
    g = np.random.default_rng(seed)
    A = g.uniform(-1, 1, (M, K)).astype(np.float32)
    B = g.uniform(-1, 1, (K, N)).astype(np.float32)
    if values == "e4m3":          # exact sums, many ties and zero sums
        A, B = (oracle.virtual_round((v / 16).ravel(), (8, 3, 7, 1, 0, 0)).reshape(v.shape)
                for v in (A, B))
    elif values == "wide":        # sums that overflow, cancel and reach FP32's subnormals
        A, B = ((v * np.exp2(g.uniform(-70, 62, v.shape))).astype(np.float32) for v in (A, B))
    elif values == "tiny":        # FP32-subnormal products and operands, signed zeros
        A, B = ((v * np.exp2(g.uniform(-88, -60, v.shape))).astype(np.float32) for v in (A, B))
        A[g.random(A.shape) < 0.1] = -0.0
        B[g.random(B.shape) < 0.02] = 1e-41
    elif values == "large":       # binary16 sums in and past the top binades
        A *= 256
        B *= 64
    elif values == "special":
        for X in (A, B):
            for v in (0.0, -0.0, np.inf, -np.inf, np.nan, 1e-41, 3e38):
                X.flat[g.integers(0, X.size, 2)] = v
        A.view(np.uint32).flat[0] = 0xFFFFFFFF        # a NaN whose payload is all ones
    return A, B


def _odd_ld(x, dev):
    """x inside a larger buffer: an odd leading dimension, first element not 16-byte aligned."""
    r, c = x.shape
    buf = torch.full((r + 1, c + 3 - c % 2), float("nan"), device=dev)
    buf[1:, 1:1 + c] = torch.from_numpy(x).to(dev)
    return buf[1:, 1:1 + c]


def _run(lof, A, B, acc, dev, ta, tb, config, odd):
    put = (lambda x: _odd_ld(x, dev)) if odd else (lambda x: torch.from_numpy(x).to(dev))
    Ad = put(np.ascontiguousarray(A.T)).t() if ta else put(A)
    Bd = put(np.ascontiguousarray(B.T)).t() if tb else put(B)
    return lof.gemm(Ad, Bd, acc, alpha=0.75, config=config).cpu().numpy()


@pytest.mark.parametrize("values", ["uniform", "e4m3", "wide", "tiny", "large", "special"])
@pytest.mark.parametrize("kind", [1, 10, 22, 23, HALF, HALF_EXT, HALF_WIDE], ids=str)
def test_accumulators_and_values(dev, kind, values):
    import lofloat_amd as lof
    M, N, K = 33, 70, 131
    A, B = _operands(M, N, K, values, seed=11)
    for chunk in (1, 2, 4, 8, 16, 32):
        acc, oacc = _accums(lof, kind, chunk)
        ref = oracle.gemm(A, B, oacc, alpha=0.75)
        for cfg in CONFIGS:
            got = _run(lof, A, B, acc, dev, False, True, cfg, cfg % 2 == 0)
            assert_bits(got, ref, f"{kind} {values} chunk {chunk} config {cfg}")


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 130, 33), (15, 64, 128), (16, 65, 129),
                                   (17, 16, 127), (64, 17, 64), (65, 63, 31), (129, 127, 65),
                                   (130, 131, 96)], ids=str)
@pytest.mark.parametrize("odd", [False, True])
def test_edges_and_layouts(dev, shape, odd):
    import lofloat_amd as lof
    M, N, K = shape
    A, B = _operands(M, N, K, "uniform", seed=M + N + K)
    for kind, chunk in ((10, 8), (HALF, 32), (23, 4), (7, 1), (HALF, 1), (23, 1)):
        acc, oacc = _accums(lof, kind, chunk)
        ref = oracle.gemm(A, B, oacc, alpha=0.75)
        for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
            for cfg in (-1, *CONFIGS):
                assert_bits(_run(lof, A, B, acc, dev, ta, tb, cfg, odd), ref,
                            f"{shape} {kind} chunk {chunk} ta {ta} tb {tb} config {cfg}")


@pytest.mark.parametrize("chunk", [1, 8, 32])
@pytest.mark.parametrize("case", [(3, 20, 9, 9, 3, 1, 1), (2, 5, 13, 70, 3, 2, 1),
                                  (1, 33, 17, 130, 1, 1, 0), (2, 3, 20, 24, 7, 2, 3)], ids=str)
def test_conv(dev, case, chunk):
    import lofloat_amd as lof
    batch, cin, size, cout, k, stride, pad = case
    g = np.random.default_rng(5)
    x = g.uniform(-1, 1, (batch, cin, size, size)).astype(np.float32)
    w = g.uniform(-1, 1, (cout, cin, k, k)).astype(np.float32)
    for kind in (10, 23, HALF):
        acc, oacc = _accums(lof, kind, chunk)
        ref = oracle.conv2d(x, w, oacc, pad=(pad, pad), stride=(stride, stride))
        for cfg in (-1, 6, 7):
            y = lof.conv2d(torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), acc,
                           stride=stride, padding=pad, config=cfg).cpu().numpy()
            assert_bits(y, ref, f"conv {case} {kind} chunk {chunk} config {cfg}")


@pytest.mark.parametrize("bits", [10, 23, HALF], ids=str)
@pytest.mark.parametrize("case", ["grows", "mixed", "zeros", "one_bit", "columns", "zero_a"])
def test_chunk_1_leaf_changes(dev, case, bits):
    """Chunk 1, 23 bits: slices whose sums are all exact run on the MFMA, the others leaf by leaf,
    and a wave goes from one to the other as its accumulators grow (24 bits are passed about
    half way), as columns of 24-bit values come in, over zero sums of both signs, and with one
    inexact term in an otherwise exact product.  10 bits: from the packed binary16 leaves on the
    grid to the checked and the directed ones and back, with columns 2^40 apart in a wave and a
    zero operand slice beside large values.  Binary16: from packed slices to FP32 ones where a value
    is no binary16 one."""
    import lofloat_amd as lof
    M, N, K = 70, 66, 520
    g = np.random.default_rng(31)
    A, B = (oracle.virtual_round(g.standard_normal(s).astype(np.float32).ravel(),
                                 (8, 3, 7, 1, 0, 0)).reshape(s) for s in ((M, K), (K, N)))
    if case == "grows":
        A, B = np.abs(A) * 8, np.abs(B) * 8 + np.float32(2.0 ** -9)
    elif case == "mixed":
        A[:, 200:230] = g.standard_normal((M, 30)).astype(np.float32)
    elif case == "zeros":
        A[:, 1::2] = -A[:, ::2]
        B[1::2] = B[::2]
        A[3] = -0.0
    elif case == "columns":
        A = g.uniform(-1, 1, (M, K)).astype(np.float32)
        B[:, ::7] *= np.float32(2.0 ** 40)
    elif case == "zero_a":
        A[:, 64:192] = 0.0
        B[64:192] *= np.float32(2.0 ** 30)
    else:
        A[5, 300] = np.float32(1 + 2.0 ** -23)
    acc, oacc = _accums(lof, bits, 1)
    ref = oracle.gemm(A, B, oacc, alpha=0.75)
    for cfg in CONFIGS:
        for ta, tb in ((0, 1), (1, 0)):
            assert_bits(_run(lof, A, B, acc, dev, ta, tb, cfg, False), ref, f"{case} config {cfg}")


@pytest.mark.parametrize("scale", [0, 20, 60, 110, -60, -75])
def test_mfma_is_the_fmaf_chain(dev, scale):
    """23-bit chunk-32 sums of one chunk, on the f32 MFMA against the VALU fmaf chain (config
    bit 0x200), over operand magnitudes from FP32's subnormal products to overflow."""
    import lofloat_amd as lof
    g = torch.Generator(device=dev).manual_seed(scale + 100)
    acc = lof.AccumSpec(mant_bits=22, chunk=32)
    spread = abs(scale) if scale < 100 else 12
    for rep in range(4):
        A, B = ((torch.rand(2048, 32, device=dev, generator=g) * 2 - 1) *
                torch.exp2(torch.randint(-spread, 1, (2048, 32), device=dev, generator=g) / 2 +
                           (scale / 2 if scale != 0 else 0)) for _ in range(2))
        ref = lof.gemm(A, B.t(), acc, config=7 | 0x200)
        for cfg in (7, 9):
            got = lof.gemm(A, B.t(), acc, config=cfg)
            same = (got.view(torch.int32) == ref.view(torch.int32)) | (got.isnan() & ref.isnan())
            assert bool(same.all()), (scale, rep, cfg, int((~same).sum()))
