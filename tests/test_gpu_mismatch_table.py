"""The all-mismatch table at sizes around its strips (64 and 256 rows, blocks of
16 columns), the empty one and the largest, against the oracle's."""
import numpy as np
import pytest

import oracle as O
from gat_amd import _native as N

from tests.devbuf import DevBuf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxlen", [0, 1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1000, 2047, 2048])
def test_mismatch_table_sizes(gpu, maxlen):
    w = maxlen + 1
    out = DevBuf.of(np.full(w * w + 64, -7, np.int32))
    N.check_hip(N.hip().gat_edr_mismatch_table(maxlen, out.ptr, None))
    got = out.get(np.int32, w * w + 64)
    assert (got[:w * w].reshape(w, w) == O.ftable(maxlen)).all()
    assert (got[w * w:] == -7).all()
