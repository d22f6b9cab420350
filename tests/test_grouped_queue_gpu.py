"""GPU checks of the grouped launch's work queue and of the config it picks."""
import numpy as np
import pytest
import torch

import oracle
from conftest import assert_bits

pytestmark = pytest.mark.gpu

HALF, BF16 = (16, 10, 15, 1, 0, 0), (16, 7, 127, 1, 0, 0)


def _fmt(t):
    import lofloat_amd as lof
    return lof.FloatFormatDescriptor(*t, lof.formats.P3109_InfChecker(t[0]),
                                     lof.formats.P3109_NaNChecker(t[0]))


def _accum(kind, chunk):
    import lofloat_amd as lof
    if isinstance(kind, int):
        return lof.AccumSpec(mant_bits=kind, chunk=chunk), oracle.accum_mant(kind, chunk)
    return lof.AccumSpec(fmt=_fmt(kind), chunk=chunk), oracle.accum_fmt(kind, chunk)


def test_tuned_config_only_where_it_takes_the_products(dev):
    """The tuned config applies to later plans, but the one of the chunk-sum kernels not to a plan with
    chunk sums that they do not take (a bfloat16-shaped accumulator): its VALU tile would run them."""
    import lofloat_amd as lof
    jobs = [lof.GemmJob(torch.randn(256, 256, device=dev), torch.randn(256, 256, device=dev),
                        _accum(HALF, 8)[0]) for _ in range(24)]
    tuned, _ = lof.grouped.autotune(jobs, iters=3)
    assert lof.GroupedPlan(jobs).info()[0] == lof.GroupedPlan(jobs, config=tuned).info()[0]
    other = [lof.GemmJob(torch.randn(256, 256, device=dev), torch.randn(256, 256, device=dev),
                         _accum(BF16, 32)[0])]
    last = lof.grouped.num_configs() - 1
    assert lof.grouped.config_name(last).endswith("mfma32x32")
    picked, on_valu = (lof.GroupedPlan(other, config=c).info()[0] for c in (-1, last))
    assert picked != on_valu and picked in (4 * 4, 2 * 4), (tuned, picked, on_valu)


def _gemm_jobs(dev, seed):
    """Products of every accumulator kind at chunk 1, and of the chunk sums, with their oracle results."""
    import lofloat_amd as lof
    g = np.random.default_rng(seed)
    jobs, refs = [], []
    for i, (kind, chunk) in enumerate([(7, 1), (10, 1), (23, 1), (HALF, 1), (23, 8), (10, 16), (HALF, 32),
                                       (7, 8), (BF16, 1), (BF16, 4), (23, 3)]):
        M, N, K = (int(v) for v in g.choice([33, 64, 70, 129], 3))
        A, B = (g.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N)))
        if i % 3 == 2:
            A, B = (oracle.virtual_round(v.ravel(), (8, 3, 7, 1, 0, 0)).reshape(v.shape) for v in (A, B))
        acc, oacc = _accum(kind, chunk)
        Bd = torch.from_numpy(np.ascontiguousarray(B.T)).to(dev).t() if i % 2 else torch.from_numpy(B).to(dev)
        jobs.append(lof.GemmJob(torch.from_numpy(A).to(dev), Bd, acc, alpha=0.75))
        refs.append(oracle.gemm(A, B, oacc, alpha=0.75))
    return jobs, refs


@pytest.mark.parametrize("config", range(-1, 9))
def test_more_tiles_than_workgroups(dev, config):
    """Several times the tiles that the grid has workgroups: the first of each comes by index, the others
    from the counter, which the launch leaves at zero -- launched, replayed and run without
    allocation several times, with every output checked each time."""
    import lofloat_amd as lof
    assert lof.grouped.num_configs() == 9
    jobs, refs = _gemm_jobs(dev, 5 + config)
    g = torch.Generator(device=dev).manual_seed(config + 1)
    big = []
    for i in range(4):
        x = torch.randn(8_000_000 + 4321 * i, device=dev, generator=g)
        if i % 2:
            x = x[:x.numel() // 32 * 32]
            big.append((lof.MXJob(x, 32, _fmt((8, 3, 7, 1, 0, 0)), lof.create_e8m0_params()),
                        lof.virtual_mx_round(x, 32, _fmt((8, 3, 7, 1, 0, 0)), lof.create_e8m0_params())))
        else:
            big.append((lof.RoundJob(x, 5 + i), lof.virtual_round(x, 5 + i)))
    every = jobs + [j for j, _ in big]
    plan = lof.GroupedPlan(every, config=config)
    tiles, grid = plan.info()
    assert tiles > 2 * grid, (tiles, grid)
    graph = plan.capture_graph()
    for rep in range(4):
        for name, run in (("plan", plan.run), ("graph", graph.replay),
                          ("no allocation", lambda: lof.grouped.run_noalloc(every, config=config))):
            for j in every:
                j.out.fill_(float("nan"))
            run()
            torch.cuda.synchronize()
            for j, r in big:
                assert torch.equal(j.out.view(torch.int32), r.view(torch.int32)), (name, rep)
            for k, (j, r) in enumerate(zip(jobs, refs)):
                assert_bits(j.out.cpu().numpy(), r, f"{name} rep {rep} job {k}")
