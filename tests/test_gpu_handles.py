"""Many handles at once: each has its own place for the norms that the GPU
writes to host memory, whichever thread made it and whatever handles were
destroyed before.  More handles than one page of such places holds, norms taken
from four threads, equal bit for bit to those of one handle that is given each
state in turn."""
import threading

import numpy as np
import pytest

from festgpu import cases as C
from festgpu.native import GpuBlock

pytestmark = pytest.mark.gpu
N, THREADS = 280, 4


def test_norms_of_many_handles():
    case, nodes, q = C.euler_bump(6, 5, 4)

    def state(n):
        s = q.copy()
        s[1:4, 3:-3, 3:-3, 3:-3] *= 1 + 1e-3 * (n + 1)
        return s

    def block(n):
        g = GpuBlock(case)
        g.set_grid(nodes)
        g.upload_state(state(n))
        g.residual(1)
        return g

    one = block(0)
    want = []
    for n in range(N):
        one.upload_state(state(n))
        one.residual(1)
        want.append(one.resnorm())
    assert len({w.tobytes() for w in want}) == N

    blocks, got = [None] * N, [None] * N

    def run(what):
        errors = []

        def work(t):
            try:
                for n in range(t, N, THREADS):
                    what(n)
            except Exception as e:  # a thread's failure is the test's
                errors.append((t, e))
        threads = [threading.Thread(target=work, args=(t,)) for t in range(THREADS)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors

    def make(n):
        if blocks[n] is None:
            blocks[n] = block(n)

    def norms(n):
        got[n] = blocks[n].resnorm()

    def drop(n):
        if n % 3:
            blocks[n].close()
            blocks[n] = None

    for _ in range(2):
        run(make)
        run(norms)
        for n in range(N):
            assert np.array_equal(got[n], want[n]), n
        run(drop)
    for g in blocks:
        if g is not None:
            g.close()
