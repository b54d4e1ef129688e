"""The generated kernels' static LDS stays within the 160 KB of a compute unit for any number of
polarisations: the wave groups' exchange buffers grow with it, so models with many get fewer
groups."""
import re

import pytest

from helpers import plan_of
from ctpwa_amd import _native
from ctpwa_amd import workloads as W


@pytest.mark.parametrize("npol", [2, 9, 10, 20, 21, 64])
def test_static_lds_fits(npol):
    pol = "polarization: [" + ", ".join(["1", "0", "-1"][k % 3] for k in range(npol)) + "]"
    text = plan_of(W.JPSI_KKPIPI_WIDE.replace("polarization: [1, -1]", pol)).to_text()
    assert "npol %d " % npol in text
    size = {"double": 8, "unsigned char": 1}
    for precision in ("fp64", "mixed"):
        for src in (_native.generate_source(text, precision), _native.generate_hessian_source(text, precision)):
            kernels = re.split(r'extern "C" __global__', src)[1:]
            assert kernels
            for k in kernels:
                lds = 8
                for t, dims in re.findall(r"__shared__ (?:__attribute__\(\(aligned\(16\)\)\) )?(double|unsigned char) \w+((?:\[\d+\])+)", k):
                    n = size[t]
                    for d in re.findall(r"\d+", dims):
                        n *= int(d)
                    lds += n
                assert lds <= 160 * 1024, (npol, precision, lds)
