"""forward_many refuses rows of another width before the library reads them (CPU)."""
import types

import numpy as np
import pytest

from tdscha_amd.terminator import forward_many


@pytest.mark.parametrize("rows, dims", [((4, 79), [[80, 10]]), ((4, 81), [[80, 10]]),
                                        ((79,), [[80, 10]]), ((4, 80), [[80, 10], [60, 10]]),
                                        ((4, 80), [[80, 10], [80, 9]]), ((4, 80), [])])
def test_rows_of_another_width(rows, dims):
    nets = [types.SimpleNamespace(dims=d, shape=(d[0], 1, 0, d[-1]), h=None) for d in dims]
    with pytest.raises(ValueError):
        forward_many(nets, np.zeros(rows, np.float32))
