"""Colour passes with every workgroup size give the same bits on a box of
each band of the default's rule (launches of up to 100,000 threads, some
hundred thousand, and a million), in FP64, mixed precision and for
Punctures_EM (one point a thread)."""
import numpy as np
import pytest

import ollipticid_amd as oa
from tests.test_gpu_norms import EM
from tests.test_gpu_vector_paths import argv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order", [(33, 4), (97, 2), (129, 8), (161, 2)])
@pytest.mark.parametrize("kind", ["fp64", "mixed", "em"])
def test_sizes_give_the_same_bits(kind, n, order):
    a = EM + ["-N", str(n), "-O", str(order)] if kind == "em" else argv(0, n, order)
    p = oa.problem_from_argv(a)
    p.precision = oa.PREC_MIXED if kind == "mixed" else oa.PREC_FP64
    print("case", kind, n, order, flush=True)
    before = oa.sweep_threads(p.precision, order)
    rng = np.random.default_rng(n)
    with oa.Hierarchy(p) as h:
        try:
            top = h.levels - 1
            ib = h.nbox - 1
            u = 1.0 + 1e-2 * rng.standard_normal(h.boxes()[ib]["n"][::-1])
            runs = {}
            for threads in (256, 64, 128, 512):
                oa.set_sweep_threads(p.precision, order, threads)
                h.set_field(ib, oa.F_U, u)
                norm = h.smooth(top, 2)
                runs[threads] = norm, h.get_field(ib, oa.F_U)
            for threads, (norm, field) in runs.items():
                assert norm == runs[256][0], threads
                assert np.array_equal(field, runs[256][1]), threads
        finally:
            oa.set_sweep_threads(p.precision, order, before)
