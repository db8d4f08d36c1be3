"""affine quantize: values where the short path's divisions, clamps and packing could
differ from the reference's arithmetic, and groups that must leave it."""
import pytest
import torch

from tests.test_gpu_quantize import _check_quantize
from tests.util import ALL_BITS, ALL_GROUPS, DTYPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bits", ALL_BITS)
@pytest.mark.parametrize("gs", ALL_GROUPS)
def test_ties_extremes_and_mixed_waves(oracle, gpu, dtype, bits, gs):
    g = torch.Generator().manual_seed(bits + gs)
    big = 3.0e4 if dtype == torch.float16 else 1e31
    rows = []
    # quotients at and next to halves: few mantissa bits, symmetrical and one-sided groups
    for lo, hi in ((-8, 8), (-15, 16), (1, 33), (-64, -3), (0, 2)):
        rows.append(torch.randint(2 * lo, 2 * hi + 1, (1024,), generator=g).float() / 2)
    rows.append(torch.randn(1024, generator=g) * 1e-3 + 7.0)      # far from zero, narrow
    rows.append(torch.randn(1024, generator=g) * 2e-5)            # about the range 1e-4
    rows.append(torch.randn(1024, generator=g) * big / 4)         # past 1e30 where it fits
    mixed = torch.randn(1024, generator=g)                        # one odd group in a wave
    mixed[256:256 + gs] = 0.0
    rows.append(mixed)
    spike = torch.randn(1024, generator=g) * 1e-6
    spike[::gs] = 5.0
    rows.append(spike)
    _check_quantize(oracle, gpu, torch.stack(rows).to(dtype), gs, bits)
