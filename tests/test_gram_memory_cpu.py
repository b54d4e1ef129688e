"""Device memory of the amplitude Gram that a handle without free resonance parameters keeps:
its rows take at most 256 MiB whatever the number of events, and with the weights, the sums of
the tile pairs and the result the 149-amplitude model's workspace stays below 340 MiB."""
import re

import pytest

from helpers import plan_of
from ctpwa_amd import _native
from ctpwa_amd import workloads as W


@pytest.mark.parametrize("n", [50_000, 500_000, 10_000_000])
@pytest.mark.parametrize("precision", [0, 1])
def test_rows_of_the_stored_gram_are_bounded(n, precision):
    free = plan_of("jpsi_kkpipi_wide").to_text()
    fixed = plan_of(re.sub(r", +free: \[[^\]]*\]", "", W.JPSI_KKPIPI_WIDE)).to_text()
    f = _native.lib().ctpwa_footprint_bytes
    extra = f(fixed.encode(), n, n // 5, 0, precision) - f(free.encode(), n, n // 5, 0, precision)
    assert 0 < extra <= 340 << 20
