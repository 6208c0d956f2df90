"""Creating a context does not wait for the work of another one."""
import ctypes
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_context_creation_beside_a_running_lattice(kmi, backend):
    from kraken_mi355x import _lib as L

    lib = L.load()
    with kmi.Lattice(kmi.make_desc("d3q19", 256, 256, 256, 0.02, storage="f64", collision="trt"), backend) as lat:
        lat.set_temporal(0)
        lat.step(3)
        started, done = threading.Event(), threading.Event()

        def run():
            started.set()
            lat.step(1000)  # about a second; creating a context takes a few milliseconds
            done.set()

        t = threading.Thread(target=run)
        t.start()
        started.wait()
        while lat.steps == 3:  # the run's launches are queued
            pass
        ctx = ctypes.c_void_p()
        rc = lib.kmi_ctx_create(0, ctypes.byref(ctx))
        overlapped = not done.is_set()
        t.join()
        assert rc == 0
        lib.kmi_ctx_destroy(ctx)
        assert overlapped
