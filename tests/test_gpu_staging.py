"""Field and point exchange with the host where no pinned memory is to be had
(the allocation is made to fail on the host): the same bits."""
import ctypes as C

import numpy as np
import pytest

import ollipticid_amd as oa
from tests.test_gpu_vector_paths import argv

pytestmark = pytest.mark.gpu


class NoPinned:
    """The pool drained and its allocator failing."""

    def __enter__(self):
        self.L = oa.load()
        self.take = getattr(self.L, "_ZN3oll12staging_takeEi")
        self.take.restype, self.take.argtypes = C.c_void_p, [C.c_int]
        self.give = getattr(self.L, "_ZN3oll12staging_giveEPNS_7StagingE")
        self.give.restype, self.give.argtypes = None, [C.c_void_p]
        self.hook = C.c_void_p.in_dll(self.L, "_ZN3oll14staging_mallocE")
        self.saved = self.hook.value
        self.calls = 0

        def fail(p, n, flags):
            self.calls += 1
            return 2  # hipErrorOutOfMemory

        self.fail = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_size_t, C.c_uint)(fail)
        self.hook.value = C.cast(self.fail, C.c_void_p).value
        self.held = []
        while True:
            s = self.take(1)
            if not s:
                break
            self.held.append(s)
        self.calls = 0
        return self

    def __exit__(self, *exc):
        self.hook.value = self.saved
        for s in self.held:
            self.give(s)


@pytest.mark.parametrize("n,order", [(25, 2), (33, 8), (97, 4)])
def test_exchange_without_pinned_memory(n, order):
    rng = np.random.default_rng(n)
    print("case", n, order, flush=True)
    with oa.Hierarchy(oa.problem_from_argv(argv(0, n, order))) as h:
        ib = h.nbox - 1
        b = h.boxes()[ib]
        a = rng.standard_normal(b["n"][::-1])
        lo, hi = np.array(b["origin"]), np.array(b["end"])
        xyz = lo + (hi - lo) * rng.uniform(0.0, 1.0, (5000, 3))
        box = np.full(len(xyz), ib, dtype=np.int32)
        h.set_field(ib, oa.F_V, a)
        want = [h.interp(oa.F_V, box[:q], xyz[:q], 5) for q in (1, 64, 5000)]
        with NoPinned() as no:
            h.set_field(ib, oa.F_V, np.zeros_like(a))
            h.set_field(ib, oa.F_V, a)
            assert np.array_equal(h.get_field(ib, oa.F_V), a)
            for q, w in zip((1, 64, 5000), want):
                assert np.array_equal(h.interp(oa.F_V, box[:q], xyz[:q], 5), w), q
            assert no.calls >= 6  # every call went without
            assert h.residual(h.levels - 1) >= 0.0  # no error is left behind
        assert np.array_equal(h.get_field(ib, oa.F_V), a)


def test_point_calls_leave_the_budget_alone():
    """A hierarchy that fills an engine's budget is admitted again after a
    call of many points on it."""
    p = oa.problem_from_argv(argv(0, 25, 2))
    p.max_cycles = 2
    h = oa.Hierarchy(p)
    built = h.device_bytes()
    e = oa.Engine(hbm_budget=built)
    try:
        for tag in (1, 2):
            assert e.admit_hier(h, tag), tag
            while e.step():
                pass
            (_, _, _, h), = e.pop_hier({tag: p})
            b = h.boxes()[-1]
            xyz = np.random.default_rng(3).uniform(b["origin"], b["end"], (5000, 3))
            h.interp(oa.F_U, np.full(5000, h.nbox - 1), xyz, 4)
            assert h.device_bytes() >= built
        assert e.admit_hier(h, 3)
    finally:
        e.close()
