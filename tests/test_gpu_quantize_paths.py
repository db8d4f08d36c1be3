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


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bits", ALL_BITS)
@pytest.mark.parametrize("gs", ALL_GROUPS)
def test_small_groups(oracle, gpu, dtype, bits, gs):
    """Ranges and edges about eps = 1e-7 and its multiples, far below it, constants, zeros of
    both signs: the short way's form for them, bit for bit."""
    g = torch.Generator().manual_seed(bits + gs)
    n = 1 << 15
    unit = torch.randn((n // gs, gs), generator=g)
    power = torch.rand((n // gs, 1), generator=g)
    near = torch.randint(1, 8, (n // gs, 1), generator=g) * 0.5e-7 * (1 + (power - 0.5) * 1e-3)
    rows = [
        unit * 10.0 ** (-12 * power),                                  # 1 .. 1e-12
        unit * 10.0 ** (-45 + 8 * power),                              # about the end of fp32
        unit.sign() * near,                                            # edges of some half eps
        near + unit * 1e-9,
        torch.where(unit > 0, near * (2 ** bits - 1), near * 0.0),     # ranges of some n_bins eps
        near.expand_as(unit) * 1e7,                                    # constants
        unit * 0.0,
        torch.where(power < 0.3, unit * 0.0, unit),                    # some groups pruned
    ]
    w = torch.stack([r.reshape(-1) for r in rows]).to(dtype)
    _check_quantize(oracle, gpu, w, gs, bits)
