"""IrLP on both sides of the vertex count from which a wave stages its rows
entry by entry: labels bit for bit against the oracle, with rows that fill a
wave's stage and rows past it."""
import numpy as np
import pytest

import labelpropcuda_amd as L
import oracle.oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,degree", [(65, 3), (1000, 15), (1000, 17), (4097, 7),
                                      (1 << 20, 3), ((1 << 20) + 1, 3)])
def test_irlp_sizes(gpu_available, n, degree):
    inp = L.generate(n, degree, 3, n % 97)
    rp, ci, vv, st, gt, lab = O.irlp_final_state(inp)
    want, iters = O.irlp(rp, ci, vv, lab, st, gt, 1e-4, 9)
    got, used, _ = L.dynlp.irlp(rp, ci, vv, lab, st, gt, 1e-4, 9)
    assert used == iters
    assert np.array_equal(got.view(np.int32), np.ascontiguousarray(want, np.float32).view(np.int32))
