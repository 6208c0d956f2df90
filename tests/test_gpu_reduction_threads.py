"""Reductions of two lattices of one context from two threads: each thread gets its own lattice's sums,
the same bits as alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_two_threads_reduce_two_lattices(kmi, backend):
    # up to 16 work-groups (one launch) and more (two launches)
    for shapes in (((40, 40), (50, 61)), ((300, 200), (411, 97)), ((30, 30), (500, 400))):
        print(f"[threads] {shapes}", flush=True)
        lats = [kmi.Lattice(kmi.make_desc("d2q9", *s, 1, 0.05), backend) for s in shapes]
        for k, (lat, s) in enumerate(zip(lats, shapes)):
            r = np.random.default_rng(k)
            lat.init_equilibrium(1 + 0.02 * r.uniform(-1, 1, s), 0.02 * r.uniform(-1, 1, s), 0.02 * r.uniform(-1, 1, s))
        kinds = ("mass", "kinetic_energy", "max_speed")
        alone = [[lat.reduce(k) for k in kinds] for lat in lats]
        wrong = [0, 0]

        def work(i):
            for _ in range(400):
                wrong[i] += [lats[i].reduce(k) for k in kinds] != alone[i]

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for lat in lats:
            lat.close()
        assert wrong == [0, 0], shapes
