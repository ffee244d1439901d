"""Grouping of long tiles by four waves: chunks beyond the first 2048 rows, tiles
and chunks cut short, every compiled group count, with and without values."""
import numpy as np
import pytest

from test_gpu_grouping import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,T,G,p", [(513, 33, 512, 2, 0.1), (1100, 70, 600, 1, 0.3),
                                             (5000, 40, 4500, 2, 0.02), (2049, 100, 2049, 3, 0.05),
                                             (700, 64, 65536, 4, 0.01), (4096, 32, 2048, 2, 0.0),
                                             (1500, 31, 1024, 7, 0.1)])
@pytest.mark.parametrize("values", [False, True])
def test_long_tiles(oracle, bws, dev, rows, cols, T, G, p, values):
    rng = np.random.default_rng(rows + cols)
    D = rng.standard_normal((rows, cols)).astype(np.float32) * (rng.random((rows, cols)) < p)
    run_case(oracle, bws, dev, D.astype(np.float32), T, G, values)
