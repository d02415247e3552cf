"""The norms of the operator calls on a u that holds NaN: max |N(u)| over the
points where N(u) is a number, whichever lanes of a wave hold the others."""
import numpy as np
import pytest

import ollipticid_amd as oa
from tests.test_gpu_vector_paths import argv

pytestmark = pytest.mark.gpu

EM = ["-eq", "Punctures_EM", "-B", "Robin", "-NumBH", "1", "-bhmp1", "0.5", "-bhqp1", "0.2",
      "-bhx1", "0.3", "-L", "20", "-l", "2"]


@pytest.mark.parametrize("order", [2, 8])
@pytest.mark.parametrize("eq", [0, 1, 4])
@pytest.mark.parametrize("where", ["plane", "point"])
def test_operator_norm_beside_nan(eq, order, where):
    """A NaN in every row (a plane x = const of u) or in one point.  N(u) is
    read back whole, so the norm is its own points' exact maximum."""
    a = EM + ["-N", "33", "-O", str(order)] if eq == 4 else argv(eq, 33, order)
    print("case", eq, order, where, flush=True)
    with oa.Hierarchy(oa.problem_from_argv(a)) as h:
        rng = np.random.default_rng(5)
        boxes = h.boxes()
        for lv in range(h.levels):
            members = [ib for ib, b in enumerate(boxes) if b["level"] == lv]
            for ib in members:
                n = boxes[ib]["n"]
                u = 1.0 + 1e-2 * rng.standard_normal(n[::-1])
                if where == "plane":
                    u[:, :, n[0] // 2] = np.nan
                else:
                    u[n[2] // 2, n[1] // 2, n[0] // 2] = np.nan
                h.set_field(ib, oa.F_U, u)
            for call in (h.operator, h.residual):
                got = call(lv)
                want = 0.0
                for ib in members:
                    R = boxes[ib]["R"]
                    r = h.get_field(ib, oa.F_R)[R:-R, R:-R, R:-R]
                    assert np.isnan(r).any() and np.isfinite(r).any()
                    want = max(want, float(np.nanmax(np.abs(r))))
                assert got == want > 0.0, (lv, got, want)
