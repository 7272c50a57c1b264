"""The glue between the quantized products on the GPU against the C oracle,
bit for bit: the vision projector's exact-erf GELU (dnx_gelu,
lib/src/vision_encoder.dart:260-263, :496-509: Abramowitz-Stegun erf in
double, rounded once to float) at every start offset within a 16-byte line
and at counts around its four-values-per-thread passes, with the special
values the formula meets (signed zeros, subnormals, values whose
exponential underflows, infinities and NaN; NaN results compared as NaN)."""

import numpy as np
import pytest
import torch

from dianoia_amd import device as D
from gpu_util import bits, dev, host

pytestmark = pytest.mark.gpu

SPECIAL = np.array([0.0, -0.0, 1e-40, -1e-40, 1e-7, -1e-7, 0.5, -0.5, 3.0, -3.0, 10.0, -10.0,
                    40.0, -40.0, 1e30, -1e30, np.inf, -np.inf, np.nan], np.float32)


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 7, 8, 1023, 4099, 1 << 20])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
def test_gelu_bit_exact_at_any_offset(gpu_ready, orc, count, offset):
    rng = np.random.default_rng(count * 4 + offset)
    x = (rng.standard_normal(count) * 2).astype(np.float32)
    x[:min(count, SPECIAL.size)] = SPECIAL[:min(count, SPECIAL.size)]
    pad = np.full(offset + count + 5, 7.0, np.float32)   # guard values around x
    pad[offset:offset + count] = x
    d = dev(pad)
    D.gelu(d[offset:offset + count])
    out = host(d)
    want = orc.gelu(x)
    got = out[offset:offset + count]
    # NaN results (from NaN and -inf) are compared as NaN: their payload
    # bits are the hardware's, not the formula's.
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(bits(got[~nan]), bits(want[~nan]))
    assert np.all(out[:offset] == 7.0) and np.all(out[offset + count:] == 7.0)


@pytest.mark.parametrize("low,high", [(-150, -126), (-30, 3), (3.2, 3.45), (3, 128)])
def test_gelu_bit_exact_over_magnitudes(gpu_ready, orc, low, high):
    """Both signs from the denormals to the largest floats, and closely
    around 10, where the kernel's error function stops following |v|."""
    rng = np.random.default_rng(17)
    with np.errstate(over="ignore"):
        x = np.exp2(rng.uniform(low, high, 1 << 16)).astype(np.float32)
    x[::2] *= -1
    ten = np.float32(10.0)
    x[:4] = [np.nextafter(ten, np.float32(0)), ten, np.nextafter(ten, np.float32(11)), -ten]
    d = dev(x)
    D.gelu(d)
    got, want = host(d), orc.gelu(x)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(bits(got[~nan]), bits(want[~nan]))


def test_gelu_every_float(gpu_ready):
    """All 2^32 floats against the formula as it is written, two IEEE
    divisions and the device's exp, one operation at a time in float64: the
    kernel's product with a residual step and its Newton steps give the same
    float for every input."""
    sqrt2 = torch.tensor(1.4142135623730951, dtype=torch.float64, device="cuda")
    step = 1 << 24
    for first in range(-(1 << 31), 1 << 31, step):
        x = torch.arange(first, first + step, dtype=torch.int32, device="cuda").view(torch.float32)
        v = x.double()
        z = v.abs() / sqrt2          # (a divisor that is a number would be a product)
        t = torch.ones_like(z) / (1 + 0.3275911 * z)
        poly = ((((1.061405429 * t - 1.453152027) * t + 1.421413741) * t - 0.284496736) * t
                + 0.254829592) * t
        erf = 1 - poly * torch.exp(-z * z)
        want = (0.5 * v * (1 + torch.where(v < 0, -erf, erf))).float()
        D.gelu(x)
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(x), nan), hex(first)
        differ = (x.view(torch.int32) != want.view(torch.int32)) & ~nan
        assert int(differ.sum()) == 0, (hex(first), int(differ.sum()))
