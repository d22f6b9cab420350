"""GPU checks of the GEMM kernels at the edges of what their dispatch takes: outputs past the matrix,
leading dimensions, output sizes, and which kernel a call runs on."""
import numpy as np
import pytest
import torch

import oracle
from conftest import assert_bits

pytestmark = pytest.mark.gpu

HALF = (16, 10, 15, 1, 0, 0)


def _fmt(t):
    import lofloat_amd as lof
    return lof.FloatFormatDescriptor(*t, lof.formats.P3109_InfChecker(t[0]),
                                     lof.formats.P3109_NaNChecker(t[0]))


def _best_us(run, reps=8):
    run()
    times = []
    for _ in range(reps):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        run()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b) * 1e3)
    return min(times)


def _kernels(run):
    """Names of the device kernels that run() launches, without their arguments."""
    from torch.profiler import ProfilerActivity, profile
    run()
    torch.cuda.synchronize()
    for _ in range(3):   # a profile that recorded no kernel at all is taken again
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            run()
            torch.cuda.synchronize()
        names = [e.name.split("(lofamd")[0] for e in prof.events() if "lofamd::" in e.name]
        if names:
            break
    return names


def _overflowing(M, N, K, seed):
    """Operands whose binary16 sums pass the format's top binade within a few k."""
    g = np.random.default_rng(seed)
    return ((g.uniform(0, 400, (M, K))).astype(np.float32),
            (g.uniform(-40, 400, (K, N))).astype(np.float32))


@pytest.mark.parametrize("chunk", [1, 2, 4, 8, 16, 32])
@pytest.mark.parametrize("shape", [(3, 70, 64), (20, 130, 65), (33, 17, 96), (66, 65, 64)], ids=str)
def test_overflow_at_the_matrix_edges(dev, shape, chunk):
    import lofloat_amd as lof
    M, N, K = shape
    A, B = _overflowing(M, N, K, M + chunk)
    ref = oracle.gemm(A, B, oracle.accum_fmt(HALF, chunk))
    assert np.isinf(ref).any() or np.abs(ref).max() > 32768
    Ad, Bd = torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev)
    for cfg in (-1, *range(5, 13)):
        y = lof.gemm(Ad, Bd, lof.AccumSpec(fmt=_fmt(HALF), chunk=chunk), config=cfg).cpu().numpy()
        assert_bits(y, ref, f"{shape} chunk {chunk} config {cfg}")


@pytest.mark.parametrize("chunk", [2, 8])
def test_rows_past_the_matrix_take_no_general_leaf(dev, chunk):
    """On the 64x64 tile, 3 rows of overflowing binary16 sums need at most a quarter of the general
    leaves of 64 rows (none in the tile's lower half, 3 of 16 of a lane's outputs above); rows that
    repeat the last one took as long as real ones."""
    import lofloat_amd as lof
    A, B = (torch.from_numpy(v).to(dev) for v in _overflowing(64, 20000, 128, 1))
    acc = lof.AccumSpec(fmt=_fmt(HALF), chunk=chunk)
    few = _best_us(lambda: lof.gemm(A[:3], B, acc, config=7))
    full = _best_us(lambda: lof.gemm(A, B, acc, config=7))
    assert few < 0.7 * full, (few, full)


@pytest.mark.parametrize("chunk", [1, 4, 8, 16])
@pytest.mark.parametrize("shape", [(3, 24000, 128), (24000, 16, 128)], ids=str)
def test_few_rows_that_overflow(dev, shape, chunk):
    """Binary16 sums past the top binade with few rows or columns: one general leaf a lane and k (the
    16x16 tile), where the 16x64 and 64x16 tiles take up to four (measured 1.9 to 3.2 times as long)."""
    import lofloat_amd as lof
    M, N, K = shape
    A, B = (torch.from_numpy(v).to(dev) for v in _overflowing(M, N, K, 2))
    acc = lof.AccumSpec(fmt=_fmt(HALF), chunk=chunk)
    by_default = _best_us(lambda: lof.gemm(A, B, acc))
    wide = _best_us(lambda: lof.gemm(A, B, acc, config=10 if M <= 16 else 11))
    assert by_default < 0.8 * wide, (by_default, wide)
    assert torch.equal(lof.gemm(A, B, acc).view(torch.int32),
                       lof.gemm(A, B, acc, config=7).view(torch.int32))


@pytest.mark.parametrize("accum, mode, chunk", [
    (10, 1, 8), (10, 0, 8), (0, 0, 8), (0, 0, 2), (7, 0, 1), (23, 0, 1), (10, 0, 3),
    ((16, 7, 127, 1, 0, 0), 0, 8), ((16, 7, 127, 1, 0, 0), 1, 1), (HALF, 0, 32),
    ((14, 10, 15, 1, 0, 0), 0, 1)], ids=str)
@pytest.mark.parametrize("shape", [(2048, 4096, 8), (600, 500, 40)], ids=str)
def test_a_plans_own_launches_take_the_calls_kernel(dev, shape, accum, mode, chunk):
    """A product of a grouped plan that is launched on its own runs on the kernel of its own call."""
    import lofloat_amd as lof
    M, N, K = shape
    A, B = (torch.randn(s, device=dev) for s in ((M, K), (K, N)))
    acc = lof.AccumSpec(mant_bits=accum, chunk=chunk, mode=mode) if isinstance(accum, int) else \
        lof.AccumSpec(fmt=_fmt(accum), chunk=chunk, mode=mode)
    job = lof.GemmJob(A, B, acc)
    plan = lof.GroupedPlan([job])
    own = _kernels(lambda: lof.gemm(A, B, acc))
    assert len(own) == 1
    assert _kernels(plan.run_separate) == own
    assert torch.equal(job.out.view(torch.int32), lof.gemm(A, B, acc).view(torch.int32))


WAVE = {5: "k_gemm_mfma<2, 2,", 6: "k_gemm_mfma<2, 1,", 7: "k_gemm_mfma<1, 1,", 8: "k_gemm_mfma<1, 2,"}
CHAIN = {5: "ChainTile<32, 2, 2, 2, 2,", 7: "ChainTile<32, 2, 2, 1, 1,", 9: "ChainTile<16, 2, 2,",
         10: "ChainTile<16, 1, 4,", 11: "ChainTile<16, 4, 1,", 12: "k_gemm_few<"}


@pytest.mark.parametrize("accum", [7, 10, 23, HALF, (16, 7, 127, 1, 0, 0)], ids=str)
@pytest.mark.parametrize("chunk", [1, 4, 32])
def test_a_config_runs_the_tile_it_names(dev, accum, chunk):
    import lofloat_amd as lof
    A, B = torch.randn(150, 70, device=dev), torch.randn(70, 140, device=dev)
    acc = lof.AccumSpec(mant_bits=accum, chunk=chunk) if isinstance(accum, int) else \
        lof.AccumSpec(fmt=_fmt(accum), chunk=chunk)
    ref = lof.gemm(A, B, acc).view(torch.int32)
    for cfg in range(5, 13):
        if accum == (16, 7, 127, 1, 0, 0):        # no chunk-sum kernel: the short tiles are 64x64
            want = WAVE.get(cfg, WAVE[7])
        elif chunk == 1 and accum == 7:
            want = WAVE.get(cfg) or CHAIN[cfg]
        elif chunk == 1 and cfg == 5:
            want = WAVE[5]
        else:
            want = CHAIN.get(cfg) or WAVE[cfg]
        (name,) = _kernels(lambda: lof.gemm(A, B, acc, config=cfg))
        assert want in name, (cfg, name)
        assert torch.equal(lof.gemm(A, B, acc, config=cfg).view(torch.int32), ref), cfg


@pytest.mark.parametrize("accum", [10, 23, HALF], ids=str)
@pytest.mark.parametrize("chunk", [1, 8])
def test_a_convolutions_config_runs_the_tile_it_names(dev, accum, chunk):
    import lofloat_amd as lof
    x, w = torch.randn(2, 5, 12, 12, device=dev), torch.randn(70, 5, 3, 3, device=dev)
    acc = lof.AccumSpec(mant_bits=accum, chunk=chunk) if isinstance(accum, int) else \
        lof.AccumSpec(fmt=_fmt(accum), chunk=chunk)
    ref = lof.conv2d(x, w, acc, padding=1).view(torch.int32)
    for cfg, want in ((6, "k_conv_mfma<2, 1,"), (7, "ChainTile<32, 2, 2, 1, 1,")):
        (name,) = _kernels(lambda: lof.conv2d(x, w, acc, padding=1, config=cfg))
        assert want in name, (cfg, name)
        assert torch.equal(lof.conv2d(x, w, acc, padding=1, config=cfg).view(torch.int32), ref), cfg


def _wide(x, ld, dev):
    """x with rows ld floats apart; what lies between them is never read."""
    buf = torch.empty((x.shape[0] - 1) * ld + x.shape[1], device=dev)
    v = buf.as_strided(x.shape, (ld, 1))
    v.copy_(torch.from_numpy(x))
    return v


@pytest.mark.parametrize("ld", [(1 << 22) + 1, (1 << 25) + 3])
@pytest.mark.parametrize("ta, tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_leading_dimensions(dev, ld, ta, tb):
    """Rows 16 MiB and 128 MiB apart (past 2^25 floats, offsets within a tile pass 2^32), against the
    oracle.  Chunk sums of accumulators of 20 bits and more run on the chunk-sum kernels at any distance,
    every kind up to 2^25."""
    import lofloat_amd as lof
    M, N, K = 130, 131, 129
    g = np.random.default_rng(3)
    A, B = (g.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
    Aw, Bw = (_wide(np.ascontiguousarray(x.T) if t else x, ld, dev) for x, t in ((A, ta), (B, tb)))
    Aw, Bw = (x.t() if t else x for x, t in ((Aw, ta), (Bw, tb)))
    Ac, Bc = (torch.from_numpy(np.ascontiguousarray(x.T)).to(dev).t() if t else
              torch.from_numpy(x).to(dev) for x, t in ((A, ta), (B, tb)))
    for kind, chunk in ((23, 32), (22, 8), (20, 16), (23, 1), (10, 1), (7, 4), (HALF, 1), (HALF, 8)):
        acc = lof.AccumSpec(mant_bits=kind, chunk=chunk) if isinstance(kind, int) else \
            lof.AccumSpec(fmt=_fmt(kind), chunk=chunk)
        oacc = oracle.accum_mant(kind, chunk) if isinstance(kind, int) else \
            oracle.accum_fmt(kind, chunk)
        ref = oracle.gemm(A, B, oacc)
        for cfg in (-1, *range(5, 13)):
            y = lof.gemm(Aw, Bw, acc, config=cfg).cpu().numpy()
            assert_bits(y, ref, f"ld {ld} {kind} chunk {chunk} config {cfg}")
        for cfg in (-1, 4, 8):
            job = lof.GemmJob(Aw, Bw, acc)
            lof.GroupedPlan([job], config=cfg).run()
            assert_bits(job.out.cpu().numpy(), ref, f"grouped ld {ld} {kind} chunk {chunk} {cfg}")
        (name,) = _kernels(lambda: lof.gemm(Aw, Bw, acc))
        if ld <= 1 << 25:
            assert [name] == _kernels(lambda: lof.gemm(Ac, Bc, acc))
        else:
            assert ("k_gemm_few" if kind in (20, 22, 23) and chunk > 1 else "k_gemm_mfma") in name, kind


@pytest.mark.parametrize("kind, chunk", [(10, 1), (23, 8), (HALF, 1), (HALF, 32)], ids=str)
@pytest.mark.parametrize("N", [1 << 30, (1 << 28) + 5])
def test_long_rows(dev, kind, chunk, N):
    """One row of as many outputs as 2^24 tiles of 64, or of 16, columns: each is its operand, rounded."""
    import lofloat_amd as lof
    A = torch.ones(1, 1, device=dev)
    B = torch.empty(1, N, device=dev)
    B.copy_(torch.rand(1, 1 << 20, device=dev).repeat(1, -(-N // (1 << 20)))[:, :N])
    acc = lof.AccumSpec(mant_bits=kind, chunk=chunk) if isinstance(kind, int) else \
        lof.AccumSpec(fmt=_fmt(kind), chunk=chunk)
    y = lof.gemm(A, B, acc)
    ref = lof.virtual_round(B, kind if isinstance(kind, int) else _fmt(kind))
    assert torch.equal(y.view(torch.int32), ref.view(torch.int32))
    if kind == 10:
        y = lof.gemm(A, B, lof.AccumSpec(mant_bits=10, chunk=1, mode=1))
        ref = lof.virtual_round(B, 10, 1)
        assert torch.equal(y.view(torch.int32), ref.view(torch.int32))
