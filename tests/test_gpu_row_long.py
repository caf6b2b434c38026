"""Long rows in more than 512 rows: the edges of the 3, 5, 7 and 8 vectors a
thread holds.  Bit-exact against the oracle."""

import numpy as np
import pytest

from helpers import announce, f32
from minisgl_amd.kernel import quant_per_token
from oracle import w8a8 as orc
from test_gpu_row_shapes import DEV, _rows, _x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nvec", [1536, 1537, 2560, 2561, 3584, 3585, 4096])
def test_quant_long_rows(nvec):
    announce(f"quant long rows 514 x {8 * nvec}")
    x = _x(514, 8 * nvec, nvec)
    q, s = quant_per_token(x.to(DEV))
    r = _rows(514)
    q_ref, s_ref = orc.quant_per_token(f32(x[r]))
    np.testing.assert_array_equal(q.cpu().numpy()[r], q_ref)
    np.testing.assert_array_equal(s.cpu().numpy()[r].view(np.uint32), s_ref.view(np.uint32))
