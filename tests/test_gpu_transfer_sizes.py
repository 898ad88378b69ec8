"""Fields across the host boundary on both sides of the sizes at which they are
transposed on the host, read as floats a piece at a time, or moved as doubles: what
was written comes back, and the other fields are as they were."""
import numpy as np
import pytest

import qmin

pytestmark = pytest.mark.gpu


# FP64: 16,384 sites and one row more; FP32: 65,536 and a row more, pieces of 52,429
# sites that the sites do and do not fill, 2^20 sites and a row more
@pytest.mark.parametrize("precision,shape", [(qmin.QM_FP64, (16, 32, 32)), (qmin.QM_FP64, (16, 33, 32)),
                                             (qmin.QM_FP32, (64, 32, 32)), (qmin.QM_FP32, (64, 33, 32)),
                                             (qmin.QM_FP32, (131, 51, 31)), (qmin.QM_FP32, (128, 128, 64)),
                                             (qmin.QM_FP32, (128, 129, 64))])
def test_fields_round_trip_at_the_limits(precision, shape):
    g = qmin.Lattice(*shape, precision=precision)
    rng = np.random.default_rng(shape[1])
    fields = {}
    for which in (qmin.FIELD_Q, qmin.FIELD_V, qmin.FIELD_F):
        a = rng.normal(size=(g.n, 5))
        g.set_field(which, a)
        fields[which] = a if precision == qmin.QM_FP64 else a.astype(np.float32).astype(np.float64)
    for which, a in fields.items():
        assert np.array_equal(g.get_field(which), a)
