"""Kernels that take several points of a row per thread, at the row lengths
where they can go wrong (odd and even numbers of points of a colour, rows
shorter and longer than a wave), against the oracle stage by stage; the
tolerance is test_gpu_parity's."""
import numpy as np
import pytest

import ollipticid_amd as oa
from oracle import oracle as O
from tests.test_gpu_parity import PUNC, pair, rel_err, seed_state

pytestmark = pytest.mark.gpu

SHELL = ["-eq", "Punctures_scalar_field", "-B", "Robin", "-psc", "2", "-phi0", "0.02", "-a2", "1",
         "-r0", "10", "-sigma", "4"]


def argv(eq, n, order, levels=2):
    return (PUNC if eq == 0 else SHELL) + [
        "-NumBH", "1", "-bhmp1", "0.8", "-bhx1", "0.5", "-bhy1", "-0.3", "-bhpy1", "0.15",
        "-bhsz1", "0.1", "-L", "50", "-N", str(n), "-l", str(levels), "-O", str(order), "-s", "1e-12"]


@pytest.mark.parametrize("order", [2, 4, 6, 8])
@pytest.mark.parametrize("eq,n", [(0, 25), (1, 33), (0, 41)])
def test_paired_sweeps(eq, n, order):
    h, s = pair(argv(eq, n, order))
    seed_state(h, s, 31)
    for lv in range(s.levels):
        ng = h.smooth(lv, 3)
        no = max(s.smooth(ib, 3) for ib in s.level_boxes(lv))
        assert abs(ng - no) <= 1e-11 * no, (lv, ng, no)
        for ib in s.level_boxes(lv):
            assert rel_err(h.get_field(ib, oa.F_U), s.field(ib, O.F_U)) < 1e-12, (lv, ib)
    h.close()


@pytest.mark.parametrize("eq", [0, 1])
@pytest.mark.parametrize("n", [25, 33, 41])  # coarsest boxes 13^3, 17^3, 21^3
def test_coarsest_solve(eq, n):
    """One FAS step: the coarsest box with its faces, edges and corners, and
    every finer box that reads them."""
    h, s = pair(argv(eq, n, 2))
    top = s.levels - 1
    for _ in range(2):
        ng, no = h.fas(top), s.fasn(top)
        assert abs(ng - no) <= 1e-9 * no, (ng, no)
        for ib in range(s.nbox):
            assert rel_err(h.get_field(ib, oa.F_U), s.field(ib, O.F_U)) < 1e-12, ib
    h.close()


@pytest.mark.parametrize("n,order", [(25, 2), (33, 8), (65, 4), (81, 6), (129, 2)])
def test_field_exchange(n, order):
    """A field written and read back whole, in one piece and in several (a
    half of the pinned staging holds 2^19 points), and single points of it
    through the interpolation at grid points."""
    h = oa.Hierarchy(oa.problem_from_argv(argv(0, n, order)))
    rng = np.random.default_rng(7)
    for ib in (h.nbox - 1, h.nbox - 2):
        b = h.boxes()[ib]
        a = rng.standard_normal(b["n"][::-1])
        h.set_field(ib, oa.F_V, a)
        assert np.array_equal(h.get_field(ib, oa.F_V), a)
        ijk = np.stack([rng.integers(1, b["n"][a_] - 1, 500) for a_ in range(3)], axis=1)
        xyz = np.array(b["origin"]) + ijk * np.array(b["d"])
        got = h.interp(oa.F_V, np.full(500, ib), xyz, 3)
        assert np.array_equal(got, a[ijk[:, 2], ijk[:, 1], ijk[:, 0]])
    h.close()


@pytest.mark.parametrize("order", range(1, 10))
def test_interp_orders(order):
    """Every interpolation order against the oracle, bit for bit, on both
    sides of each change of route (few points, one chunk, several)."""
    h, s = pair(argv(0, 25, 4))
    seed_state(h, s, 3)
    ib = s.nbox - 1
    b = h.boxes()[ib]
    rng = np.random.default_rng(order)
    lo, hi = np.array(b["origin"]), np.array(b["end"])
    xyz = lo + (hi - lo) * rng.uniform(0.0, 1.0, (65537 + 1000, 3))
    box = np.full(len(xyz), ib, dtype=np.int32)
    few = h.interp(oa.F_U, box[:4096], xyz[:4096], order)
    want = [s.interp(ib, O.F_U, O.I_LAGRANGE, order, *x) for x in xyz[:200]]
    assert np.array_equal(few[:200], want)
    for count in (1, 15, 17, 4097, 65536, 65537, len(xyz)):
        got = h.interp(oa.F_U, box[:count], xyz[:count], order)
        assert np.array_equal(got[:4096], few[:count])
        # the last points alone take the short route
        tail = min(count, 50)
        assert np.array_equal(got[-tail:], h.interp(oa.F_U, box[:tail], xyz[count - tail:count], order))
    h.close()
