"""Step graphs while other host threads use their own handles: a handle belongs
to one thread, several threads may work at once.  Runs long enough to build and
replay their graphs, of lone solvers and of a batch, beside a thread that sets
and reads states and creates solvers all the while: no call of either fails, the
replays take place, and the states equal those of single steps."""
import threading

import numpy as np
import pytest

import small_cases as sc
from lfm_public_amd import capi

pytestmark = pytest.mark.gpu


def test_graphs_beside_another_threads_calls():
    print("[graph threads]", flush=True)

    def case():
        return sc.vortex(16, solver=0)

    ref = capi.GpuSolver.from_case(case(), precision=capi.PREC_FP32P)
    for _ in range(400):
        ref.run(1)
    want = ref.q()
    stop, errors, rounds = threading.Event(), [], 0

    def other():
        nonlocal rounds
        try:
            while not stop.is_set():
                s = capi.GpuSolver.from_case(sc.vortex(20, solver=2, mu=0.02, minmod=1))
                q = s.q()
                for _ in range(20):
                    s.set_field(capi.FIELD_Q, q)
                    s.run(1)
                    s.field(capi.FIELD_DUDX)
                    s.field(capi.FIELD_TAUMC)
                    rounds += 1
                s.close()
        except Exception as e:  # reported by the test's thread
            errors.append(e)

    th = threading.Thread(target=other, daemon=True)
    th.start()
    try:
        for _ in range(12):
            s = capi.GpuSolver.from_case(case(), precision=capi.PREC_FP32P)
            s.run(400)
            assert np.array_equal(s.q(), want)
            assert s.replayed_steps() > 0
            s.close()
        for _ in range(6):
            members = [capi.GpuSolver.from_case(case(), precision=capi.PREC_FP32P) for _ in range(2)]
            b = capi.Batch()
            b.set(members)
            for n in (130, 270):
                b.run(n)
                b.synchronize()
            assert b.replayed_steps() > 0
            for m in members:
                assert np.array_equal(m.q(), want)
            b.close()
            for m in members:
                m.close()
    finally:
        stop.set()
        th.join(60)
    assert not errors, errors
    assert rounds > 0
    ref.close()
