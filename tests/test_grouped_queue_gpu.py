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
