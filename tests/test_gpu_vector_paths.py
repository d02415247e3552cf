"""Kernels that take several points of a row per thread, at the row lengths
where they can go wrong (odd and even numbers of points of a colour, rows
shorter and longer than a wave), against the oracle stage by stage; the
tolerance is test_gpu_parity's."""
import numpy as np
import pytest

import ollipticid_amd as oa
from oracle import oracle as O
from ollipticid_amd import native
from tests.test_gpu_parity import CASES, PUNC, pair, rel_err, seed_state

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


@pytest.mark.parametrize("case", ["o4_merge", "sf_o6", "o8", "o2_flip"])
def test_ghost_tiles_equal_points(case):
    """The ghost shells filled by tiles are those filled point by point, bit
    for bit: every order, merged boxes, tiles cut by the faces' edges."""
    out = []
    for on in (False, True):
        h = oa.Hierarchy(oa.problem_from_argv(CASES[case]))
        try:
            native.set_shared_loads(on)
            rng = np.random.default_rng(9)
            for ib, b in enumerate(h.boxes()):
                h.set_field(ib, oa.F_U, 1e-2 * rng.standard_normal(b["n"][::-1]))
            for lv in range(1, h.levels):
                h.fas(lv)
            out.append([h.get_field(ib, oa.F_U) for ib in range(h.nbox)])
        finally:
            native.set_shared_loads(True)
            h.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("order", range(2, 10))
@pytest.mark.parametrize("case", ["o4_merge", "o2_flip"])
def test_transfer_tiles(case, order):
    """Lagrange transfers against the oracle at every target point: to a
    finer level (one source box and several), to a coarser one and within a
    level, over each region, with and without `all` and `to_zero`."""
    h, s = pair(CASES[case])
    seed_state(h, s, order)
    rng = np.random.default_rng(order)
    top = s.levels - 1
    for frm, to in ((top - 1, top), (top, top - 1), (top - 2, top), (top, top)):
        for region in (0, 1, 2):
            for all_, to_zero in ((True, False), (False, False), (False, True)):
                for ib in s.level_boxes(to):
                    v = rng.standard_normal(s.field(ib, O.F_V).shape)
                    s.field(ib, O.F_V)[:] = v
                    h.set_field(ib, oa.F_V, v)
                h.transfer(frm, oa.F_U, to, oa.F_V, region, 1, order, all_, to_zero)
                s.transfer(frm, O.F_U, to, O.F_V, region, 1, order, int(all_), int(to_zero))
                for ib in s.level_boxes(to):
                    g, o = h.get_field(ib, oa.F_V), s.field(ib, O.F_V)
                    assert rel_err(g, o) < 1e-12, (frm, to, region, all_, to_zero, ib)
    h.close()


@pytest.mark.parametrize("order", [2, 4, 6, 8])
@pytest.mark.parametrize("eq,n", [(0, 25), (1, 33), (0, 41)])
def test_paired_operator(eq, n, order):
    """N(u), dN/du and the mixed-precision defect and update by two slots of
    a row a thread."""
    h, s = pair(argv(eq, n, order))
    seed_state(h, s, 32)
    for lv in range(s.levels):
        ng = h.operator(lv)
        no = max(s.residual(ib) for ib in s.level_boxes(lv))
        assert abs(ng - no) <= 1e-12 * no, lv
        for ib in s.level_boxes(lv):
            R = s.box_info(ib)["R"]
            inner = (slice(R, -R),) * 3
            assert rel_err(h.get_field(ib, oa.F_R)[inner], s.field(ib, O.F_R)[inner]) < 1e-12, (lv, ib)
    # the mixed smoothing of a linear problem (b = 0) is the FP64 one to
    # single precision: float32 sweeps of the correction, 1e-5 of it
    p = oa.problem_from_argv(argv(eq, n, order))
    p.precision = oa.PREC_MIXED
    m = oa.Hierarchy(p)
    for ib in range(s.nbox):
        u = s.field(ib, O.F_U).copy()
        m.set_field(ib, oa.F_U, u)
        h.set_field(ib, oa.F_U, u)
        if eq == 0:
            for x in (m, h):
                x.set_field(ib, oa.F_B, np.zeros_like(u))
    if eq == 0:
        for lv in range(s.levels):
            before = [h.get_field(ib, oa.F_U) for ib in s.level_boxes(lv)]
            m.smooth(lv, 2)
            h.smooth(lv, 2)
            for ib, u0 in zip(s.level_boxes(lv), before):
                a, b = m.get_field(ib, oa.F_U), h.get_field(ib, oa.F_U)
                assert np.abs(a - b).max() <= 1e-5 * np.abs(b - u0).max(), (lv, ib)
    m.close()
    h.close()


@pytest.mark.parametrize("order", [2, 4, 6, 8])
@pytest.mark.parametrize("n", [25, 41])
def test_robin_shell(n, order):
    """The Robin update of faces, edges and corners, one to four shell layers
    deep, on the smallest boxes and beside larger ones."""
    h, s = pair(argv(0, n, order))
    seed_state(h, s, 17)
    for lv in range(s.mgrid + 1):
        h.robin(lv)
        for ib in s.level_boxes(lv):
            s.robin(ib)
            assert rel_err(h.get_field(ib, oa.F_U), s.field(ib, O.F_U)) < 1e-12, (lv, ib)
    h.close()
