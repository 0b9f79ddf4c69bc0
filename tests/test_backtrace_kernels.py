"""Both backtrace kernels beside the line between them and, above it, at the edges of the 64 x 16
tiles, against the numpy restatement."""
import numpy as np
import pytest

from test_backtrace_tiles import test_backtrace_matches_numpy as matches_numpy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dtype", [(n, t) for t in (np.float32, np.float64) for n in (74, 75, 81, 84, 85, 97, 112)] +
                         [(128, np.float64), (129, np.float64)])
@pytest.mark.parametrize("cells", [0.4, 3.0])
def test_kernels_match_numpy(n, cells, dtype):
    matches_numpy(n, cells, dtype, 1e-13 if dtype == np.float64 else 2e-5)

