"""The radix sort at both edges of its tiles of 4096 records (from 2^21 records on; 2048 below)."""
import numpy as np
import pytest

from test_gpu_radix import test_coo_to_csr_matches_numpy as coo, test_transpose_is_a_stable_sort as transpose

pytestmark = pytest.mark.gpu
BIG = 2 << 20


@pytest.mark.parametrize("nnz", [2047, 2048, 2049, BIG - 2049, BIG - 1, BIG, BIG + 1, BIG + 4095, BIG + 4096, BIG + 4097])
def test_tile_edges(nnz):
    transpose(5000, 3000, nnz, True)
    coo(7000, 9000, nnz, True, np.bool_(nnz % 2))


@pytest.mark.parametrize("values", [True, False])
def test_three_passes_through_the_outputs(values):
    """More than 2^20 columns: the passes before the last go through the output arrays."""
    transpose(3000, (1 << 20) + 1, BIG + 4097, values)
    transpose(40, (1 << 24) + 3, 5000, values)
