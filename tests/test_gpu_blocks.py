"""Smoothing blocks against plain numpy: the mixed-precision block with
coefficients that matter at every point, and rows longer than a workgroup
(boxes that sixteen holes in a line merge into), which are split into
segments."""
import numpy as np
import pytest

import ollipticid_amd as oa
from tests.test_gpu_vector_paths import argv

pytestmark = pytest.mark.gpu

# second derivative: centre and the points at distance 1..R
STENCIL = {2: (-2.0, 1.0), 4: (-5 / 2, 4 / 3, -1 / 12), 6: (-49 / 18, 3 / 2, -3 / 20, 1 / 90),
           8: (-205 / 72, 8 / 5, -1 / 5, 8 / 315, -1 / 560)}


def lap(v, order, d):
    """Laplacian on the interior of v[k, j, i]."""
    R, w = order // 2, STENCIL[order]
    mid = (slice(R, -R),) * 3
    out = 0.0
    for a in range(3):
        t = w[0] * v[mid]
        for m in range(1, R + 1):
            for s in (-m, m):
                sl = list(mid)
                sl[2 - a] = slice(R + s, v.shape[2 - a] - R + s)
                t = t + w[m] * v[tuple(sl)]
        out = out + t / d[a] ** 2
    return out


class Block:
    """One box's fields and its colour order (planes k0 .. k0 + nz - 1)."""

    def __init__(self, h, ib, nz=None):
        b = h.boxes()[ib]
        self.order, self.d, self.R = b["order"], b["d"], b["R"]
        self.nc = self.R + 1
        nz = nz or b["n"][2]
        mid = (slice(self.R, nz - self.R),) + (slice(self.R, -self.R),) * 2
        names = ["b", "c", "rho"] + (["d", "e"] if h.problem.eq == 1 else [])
        ids = {"b": oa.F_B, "c": oa.F_C, "rho": oa.F_RHO, "d": oa.F_D, "e": oa.F_E}
        self.f = {q: h.get_field(ib, ids[q])[mid] for q in names}
        self.dulap = sum(STENCIL[self.order][0] / x ** 2 for x in self.d)
        k, j, i = np.indices(self.f["b"].shape, sparse=True)
        colour = (i + j + k + 3 * self.R) % self.nc
        cols = range(self.nc)
        self.masks = [colour == c for c in (reversed(cols) if b["colour_order"] else cols)]

    def op(self, u, l):
        """N(u) and dN/du from the interior u and its Laplacian."""
        f = self.f
        cu = f["c"] + u
        N = l + f["b"] * cu ** -7.0
        dN = self.dulap - 7.0 * f["b"] * cu ** -8.0
        if "d" in f:
            N = N + f["d"] * cu + f["e"] * cu ** 5.0
            dN = dN + f["d"] + 5.0 * f["e"] * cu ** 4.0
        return N, dN

    def smooth(self, u, nu):
        """u after nu FP64 sweeps, and the largest |N - rho| met."""
        u, R = u.copy(), self.R
        v = u[(slice(R, -R),) * 3]
        norm = 0.0
        for _ in range(nu):
            for m in self.masks:
                N, dN = self.op(v, lap(u, self.order, self.d))
                res = N - self.f["rho"]
                norm = max(norm, np.abs(res[m]).max())
                v[m] -= (res / dN)[m]
        return u, norm

    def correction(self, u, nu):
        """e of one mixed-precision block: nu sweeps of Lap e + q e = r."""
        R = self.R
        N, dN = self.op(u[(slice(R, -R),) * 3], lap(u, self.order, self.d))
        r, q = self.f["rho"] - N, dN - self.dulap
        e = np.zeros_like(u)
        v = e[(slice(R, -R),) * 3]
        for _ in range(nu):
            for m in self.masks:
                v[m] -= ((lap(e, self.order, self.d) + q * v - r) / (self.dulap + q))[m]
        return e


def fill(h, ib, seed, planes=None):
    """u, rho and coefficients of the size of the Laplacian's diagonal, all of
    the sign that keeps dN/du away from zero."""
    rng = np.random.default_rng(seed)
    b = h.boxes()[ib]
    n = b["n"][::-1]
    size = -sum(STENCIL[b["order"]][0] / x ** 2 for x in b["d"])

    def put(field, draw, outside=0.0):
        a = np.full(n, outside)
        a[:planes] = draw(a[:planes].shape)
        h.set_field(ib, field, a)
        return a

    u = put(oa.F_U, lambda s: 0.1 * rng.standard_normal(s).clip(-3, 3))
    put(oa.F_RHO, lambda s: size * 0.1 * rng.standard_normal(s))
    put(oa.F_C, lambda s: rng.uniform(0.9, 1.1, s), 1.0)
    put(oa.F_B, lambda s: size * rng.uniform(0.0, 0.05, s))
    if h.problem.eq == 1:
        put(oa.F_D, lambda s: -size * rng.uniform(0.0, 0.2, s))
        put(oa.F_E, lambda s: -size * rng.uniform(0.0, 0.02, s))
    return u


@pytest.mark.parametrize("order", [2, 4, 6, 8])
@pytest.mark.parametrize("eq,n", [(0, 25), (1, 33), (0, 41)])
def test_mixed_block(eq, n, order):
    """u of one block less the model's e: FP32 arithmetic of some thirty
    operations a point and two sweeps, 1e-5 of the largest e.  A wrong dN/du
    at any point shows as some 10%."""
    p = oa.problem_from_argv(argv(eq, n, order))
    p.precision = oa.PREC_MIXED
    print("case", eq, n, order, flush=True)
    with oa.Hierarchy(p) as h:
        ib = h.nbox - 1
        u = fill(h, ib, 100 * n + order)
        e = Block(h, ib).correction(u, 2)
        h.smooth(h.levels - 1, 2)
        got = h.get_field(ib, oa.F_U) - u
        assert np.abs(got - e).max() <= 1e-5 * np.abs(e).max()


def line(N, order=2):
    a = ["-eq", "Punctures", "-B", "Robin", "-NumBH", "16", "-L", "40", "-N", str(N), "-l", "2",
         "-O", str(order), "-s", "1e-10"]
    for i in range(16):
        a += ["-bhmp%d" % (i + 1), "0.3", "-bhx%d" % (i + 1), "%.6f" % ((i - 7.5) * 10.0)]
    return a


def test_rows_of_two_segments_whole_row_kernels():
    """1153 x 129 x 129 points: 289 pairs of a colour row for the operator,
    the defect and the update (256 threads), 576 points for the FP32 sweeps
    (512 threads)."""
    p = oa.problem_from_argv(line(129))
    for precision in (oa.PREC_FP64, oa.PREC_MIXED):
        p.precision = precision
        print("case: long rows", precision, flush=True)
        with oa.Hierarchy(p) as h:
            ib, top = h.nbox - 1, h.levels - 1
            assert h.boxes()[ib]["n"] == [1153, 129, 129]
            u = fill(h, ib, 7)
            m = Block(h, ib)
            if precision == oa.PREC_FP64:
                norm = h.operator(top)
                want, _ = m.op(u[1:-1, 1:-1, 1:-1], lap(u, 2, m.d))
                scale = np.abs(want).max()
                assert abs(norm - scale) <= 1e-12 * scale
                assert np.abs(h.get_field(ib, oa.F_R)[1:-1, 1:-1, 1:-1] - want).max() <= 1e-12 * scale
                norm = h.smooth(top, 1)
                after, scale = m.smooth(u, 1)
                assert abs(norm - scale) <= 1e-11 * scale
                assert np.abs(h.get_field(ib, oa.F_U) - after).max() <= 1e-12 * np.abs(after).max()
            else:
                e = m.correction(u, 1)
                h.smooth(top, 1)
                assert np.abs(h.get_field(ib, oa.F_U) - u - e).max() <= 1e-5 * np.abs(e).max()


def test_rows_of_two_segments_colour_passes():
    """2305 x 257 x 257 points: 576 pairs of a row's colour points for the
    FP64 sweeps (512 threads).  The first 16 planes are compared: one sweep
    of two colours carries a plane's values two planes on."""
    print("case: longest rows", flush=True)
    with oa.Hierarchy(oa.problem_from_argv(line(257))) as h:
        ib, top, nz = h.nbox - 1, h.levels - 1, 20
        assert h.boxes()[ib]["n"] == [2305, 257, 257]
        u = fill(h, ib, 9, planes=nz)
        after, _ = Block(h, ib, nz).smooth(u[:nz], 1)
        h.smooth(top, 1)
        got = h.get_field(ib, oa.F_U)[:16]
        assert np.abs(got - after[:16]).max() <= 1e-12 * np.abs(after).max()
