"""Lagrange transfers onto a coarser level large enough that a block takes
several chunks of points (2^21 points and more), against the oracle at every
point: covered ones, shell and untouched."""
import numpy as np
import pytest

import ollipticid_amd as oa
from oracle import oracle as O
from tests.test_gpu_parity import pair, rel_err, seed_state
from tests.test_gpu_vector_paths import argv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,region,all_,to_zero", [(3, 0, True, False), (4, 1, False, True), (9, 2, True, False)])
def test_transfer_onto_a_large_coarser_level(order, region, all_, to_zero):
    h, s = pair(argv(0, 129, 2))
    seed_state(h, s, order)
    to = h.mgrid
    (ib,) = s.level_boxes(to)
    assert np.prod(h.boxes()[ib]["n"]) >= 2 ** 21 and to + 1 < h.levels
    v = np.random.default_rng(order).standard_normal(s.field(ib, O.F_V).shape)
    s.field(ib, O.F_V)[:] = v
    h.set_field(ib, oa.F_V, v)
    h.transfer(to + 1, oa.F_U, to, oa.F_V, region, 1, order, all_, to_zero)
    s.transfer(to + 1, O.F_U, to, O.F_V, region, 1, order, int(all_), int(to_zero))
    assert rel_err(h.get_field(ib, oa.F_V), s.field(ib, O.F_V)) < 1e-12
    h.close()
    s.close()
