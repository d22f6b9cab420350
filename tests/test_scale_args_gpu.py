"""GPU checks of what the scale arguments take: everything that numpy makes one float of, and nothing
that needs a read back from the GPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [2.5, np.float64(2.5), [2.5], np.array([2.5], dtype=np.float32),
                                   torch.tensor(2.5), "2.5"], ids=repr)
@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_scales_numpy_takes(dev, scale):
    import lofloat_amd as lof
    x = torch.randn(100, device=dev)
    assert torch.equal(lof.virtual_round(x, 5, scale=scale), lof.virtual_round(x * 2.5, 5))


@pytest.mark.filterwarnings("ignore")
def test_scales_past_float_and_none(dev):
    import lofloat_amd as lof
    x = torch.ones(4, device=dev)
    assert lof.virtual_round(x, 5, scale=1e300).isinf().all()
    assert lof.virtual_round(x, 5, scale=None).isnan().all()


def test_scales_on_the_gpu_are_refused(dev):
    import lofloat_amd as lof
    one, x = torch.tensor(1.0, device=dev), torch.randn(4, 4, device=dev)
    with pytest.raises(TypeError):
        lof.virtual_round(x, 5, scale=one)
    with pytest.raises(TypeError):
        lof.lof_gemm(x, x, 10, scale_a=one, scale_b=one)
