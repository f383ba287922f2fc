"""Several threads on one handle: calls take their turns (include/tsuner.h), so
a transfer, a read of the time and the steps of an ensemble's two halves are
each whole.  Python releases the interpreter lock in every call."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from tsuner_amd import scenarios as S
from tsuner_amd.ensemble import Ensemble
from tsuner_amd.solver import Solver


def in_threads(*work):
    failed = []

    def guarded(f):
        try:
            f()
        except BaseException as e:   # a failed assertion is raised in the test's thread
            failed.append(e)

    threads = [threading.Thread(target=guarded, args=(f,)) for f in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if failed:
        raise failed[0]


def test_downloads_of_different_members():
    """FP32 members of unequal sizes (through the handle's transfer buffer,
    the largest in several pieces) and a plane, each the caller's own."""
    scs = [S.gaussian_source(n=n, dx=20.0, seed=n) for n in (40, 300, 960)]
    ens = Ensemble(scs, precision="fp32")
    want = [ens.state(i) for i in range(3)]

    def reader(i):
        def run():
            for _ in range(12):
                assert np.array_equal(ens.state(i), want[i])
                assert np.array_equal(ens.plane(i, 3), want[i][3])
        return run

    in_threads(*[reader(i) for i in (0, 1, 2, 1)])


@pytest.mark.parametrize("order", [1, 2])
def test_reads_while_an_ensemble_steps(order):
    """Members of both halves and their times, read by one thread while another
    steps: each read is the state after some whole step, and later reads are
    not of earlier steps."""
    scs = [S.gaussian_source(n=n, dx=20.0, seed=n, order=order) for n in (90, 61, 120)]
    steps = 150

    def run(visit):
        ens = Ensemble(scs, precision="fp32")
        return visit(ens)

    def alone(ens):
        out = []
        for k in range(steps + 1):
            if k:
                ens.step(1)
            out.append([(ens.plane(i, 0).tobytes(), ens.time(i)) for i in range(3)])
        return out

    want = run(alone)
    depth = [{w[i][0]: k for k, w in enumerate(want)} for i in range(3)]
    times = [{w[i][1]: k for k, w in enumerate(want)} for i in range(3)]

    def together(ens):
        def step():
            for k in (1, 2, 5, 10) * 8 + (6,):
                ens.step(k, sync=False)
            ens.synchronize()

        def read():
            seen = [0] * 3
            for j in range(40):
                i = j % 3
                k = times[i][ens.time(i)]
                assert k >= seen[i]
                seen[i] = depth[i][ens.plane(i, 0).tobytes()]
                assert seen[i] >= k

        in_threads(step, read)
        for i in range(3):
            assert ens.time(i) == want[steps][i][1]
            assert ens.plane(i, 0).tobytes() == want[steps][i][0]

    run(together)


@pytest.mark.parametrize("order", [1, 2])
def test_reads_while_a_solver_steps(order):
    """Time, dt and step number of one moment, and planes of one moment in a
    download of several pieces."""
    steps = 120
    sc = S.gaussian_source(n=960, dx=20.0, seed=3, order=order)
    a = Solver.from_scenario(sc, precision="fp32")
    want, sums = {a.time(): 0}, {a.state().sum(axis=(1, 2)).tobytes(): 0}
    for k in range(1, steps + 1):
        a.step(1)
        want[a.time()] = k
        if k % 10 == 0:
            sums[a.state().sum(axis=(1, 2)).tobytes()] = k
    b = Solver.from_scenario(sc, precision="fp32")

    def step():
        for _ in range(steps // 10):
            b.step(10, sync=False)

    def read():
        for _ in range(12):
            assert b.time() in want
            assert b.state().sum(axis=(1, 2)).tobytes() in sums

    in_threads(step, read)
    assert b.time() == a.time()
    assert np.array_equal(a.state(), b.state())
