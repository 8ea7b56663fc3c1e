"""Which kernel a call runs on, at sizes on both sides of the rules that choose it: the library's host code against a pretended HIP
runtime (tests/host/fake_hip.cpp), so that it is seen on the CPU."""
import re

import pytest


@pytest.fixture(scope="session")
def routes(host_faults):
    """(calls) -> the kernels of each, e.g. "gemm_tile_kernel<2, false, false, TileX>"."""
    def run(*calls):
        out = host_faults("routes", *calls)
        out = re.sub(r"wick_rocm::|\(anonymous namespace\)::", "", out)
        kernels = []
        for line in out.splitlines():
            if line.startswith("\t"):
                kernels[-1].append(re.sub(r"^void |\(.*$", "", line.strip()))
            else:
                kernels.append([])
        assert len(kernels) == len(calls), out
        return kernels

    return run


@pytest.mark.parametrize("dim,quads", [(32, 1), (1024, 1), (1056, 2), (2048, 2), (2080, 0), (2304, 0), (4096, 0), (8192, 0), (8224, 0)])
def test_the_norm_keeps_short_rows_only(routes, dim, quads):
    """Rows past 2048 elements are read a second time: kept, they would leave the CU four workgroups."""
    assert routes(f"norm 30 {dim}") == [[f"rmsnorm_quantize_kernel<0, {quads}>"]]
