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
