"""Which products of up to 16 rows leave the BLAS library for the weight-streaming kernel.  The sizes are those both were timed at, weights
read from memory; a side is listed where it was faster by more than 5 %.  No GPU is needed."""
import pytest

from polarquant_amd.modeling_common import _streams_faster

KERNEL = [(1, 16, 64), (8, 128, 4096), (16, 512, 4096), (8, 1024, 1024), (1, 4096, 4096), (16, 4096, 4096), (8, 3584, 3584), (1, 5120, 4096), (8, 6144, 4096),
          (8, 8192, 2048), (8, 14336, 4096), (4, 18944, 3584), (8, 32768, 2048), (1, 32768, 4096), (8, 128256, 4096), (8, 152064, 3584), (1, 4096, 14336),
          (8, 4096, 14336), (8, 3584, 18944), (8, 4096, 8192), (8, 8192, 8192), (4, 28672, 8192), (2, 8192, 28672), (8, 4096, 11008)]
LIBRARY = [(8, 128, 8192), (16, 128, 8192), (8, 256, 16384), (8, 512, 14336), (16, 512, 14336), (8, 1024, 8192), (12, 2048, 8192), (1, 16, 7168), (8, 64, 7168),
           (4, 5120, 5120), (8, 5120, 13824), (1, 4096, 16384), (1, 6144, 16384), (16, 6144, 4096), (12, 14336, 4096), (16, 32768, 4096), (9, 128256, 4096),
           (16, 152064, 3584), (9, 5120, 4096), (16, 4096, 14336), (9, 8192, 8192), (16, 8192, 4096), (12, 4608, 3584)]


@pytest.mark.parametrize("rows,n,k", KERNEL)
def test_the_kernel_takes(rows, n, k):
    assert _streams_faster(rows, n, k)


@pytest.mark.parametrize("rows,n,k", LIBRARY)
def test_the_library_keeps(rows, n, k):
    assert not _streams_faster(rows, n, k)
