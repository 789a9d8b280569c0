"""Engines of one process, and of several, that run at the same moment on a
device: a time loop is one launch (k_resident) only while no other engine's loop
is under way, and the results do not depend on what runs beside them."""
import ctypes as C
import fcntl
import os
import threading
import time

import numpy as np
import pytest

import ifos_amd
from ifos_amd import workloads

pytestmark = pytest.mark.gpu


def engine(NX, NY, NT, L=0, order=4):
    w = workloads.small_case(seed=12, NX=NX, NY=NY, NT=NT, FW=8, DTINV=4, FDORDER=order, L=L, VELOCITY=1)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)
    eng.set_shot(w.shots[0].srcpos, w.shots[0].recpos)
    return eng


def test_one_launch_only_with_the_device_to_itself(gpu_lib):
    print("[overlap] a loop beside a longer one", flush=True)
    long_, short = engine(1200, 700, 4000), engine(128, 96, 100)
    long_.set_resident(0)
    short.forward(snapshots=False)
    assert short.get_resident()[1]
    want = [np.array(x) for x in short.seismograms()]
    begun = threading.Event()

    def work():
        begun.set()
        long_.forward(snapshots=False)

    t = threading.Thread(target=work)
    t.start()
    begun.wait()
    time.sleep(0.02)  # the long loop takes over 0.1 s
    short.forward(snapshots=False)
    beside = t.is_alive()
    taken = short.get_resident()[1]
    t.join()
    assert beside and not taken
    for x, y in zip(want, short.seismograms()):
        assert np.array_equal(x, y)
    short.forward(snapshots=False)
    assert short.get_resident()[1]


def test_gradients_do_not_depend_on_what_runs_beside(gpu_lib):
    print("[overlap] three engines, ten gradients each", flush=True)
    engines = [engine(200, 90, 120, L=2, order=8), engine(400, 120, 80), engine(700, 300, 60, L=1)]
    obs = [np.random.default_rng(4).standard_normal((2,) + e.seismograms()[0].shape).astype(np.float32) for e in engines]
    want = []
    for e, o in zip(engines, obs):
        e.shot_gradient(o[0], o[1])
        want.append(np.array(e.gradient()))
    wrong = []

    def work(e, o, ref):
        for _ in range(10):
            e.shot_gradient(o[0], o[1])
            if not np.array_equal(np.array(e.gradient()).view(np.uint8), ref.view(np.uint8)):
                wrong.append(e.cfg.NX)

    threads = [threading.Thread(target=work, args=x) for x in zip(engines, obs, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_a_run_given_up_holds_back_the_other_engines(gpu_lib):
    """On a device that another process holds part of, every engine would wait
    for itself before it turned to the per-step kernels."""
    print("[overlap] a run given up", flush=True)
    first, second = engine(200, 90, 40), engine(128, 96, 40)
    first.set_resident(-1)
    first.set_resident_wait(0.0)
    first.forward(snapshots=False)
    assert not first.get_resident()[1]
    assert not second.get_resident()[0]
    second.forward(snapshots=False)
    assert not second.get_resident()[1]
    second.forward(snapshots=False)  # tried again
    assert second.get_resident() == (True, True)
    first.set_resident_wait(-1.0)
    first.forward(snapshots=False)
    assert first.get_resident() == (True, True)


def test_other_processes_loops(gpu_lib):
    """Processes lock the device's directory, shared around per-step loops and
    exclusively around a one-launch run.  (Two descriptors of one process exclude
    each other like those of two.)"""
    print("[overlap] other processes", flush=True)
    name = C.create_string_buffer(64)
    assert gpu_lib.hipDeviceGetPCIBusId(name, 64, 0) == 0
    path = "/sys/bus/pci/devices/" + name.value.decode().lower()
    if not os.path.isdir(path):
        pytest.skip("no directory of the device to lock")
    eng = engine(200, 90, 40)
    eng.set_resident(-1)
    eng.forward(snapshots=False)
    assert eng.get_resident()[1]
    want = [np.array(x) for x in eng.seismograms()]

    def run():
        t0 = time.perf_counter()
        eng.forward(snapshots=False)
        for x, y in zip(want, eng.seismograms()):
            assert np.array_equal(x, y)
        return eng.get_resident()[1], time.perf_counter() - t0

    other = os.open(path, os.O_RDONLY)
    try:
        fcntl.flock(other, fcntl.LOCK_SH)  # a per-step loop elsewhere
        taken, took = run()
        assert not taken and took < 0.2
        fcntl.flock(other, fcntl.LOCK_UN)
        assert run()[0]
        fcntl.flock(other, fcntl.LOCK_EX)  # a one-launch run elsewhere: waited for
        threading.Timer(0.05, lambda: fcntl.flock(other, fcntl.LOCK_UN)).start()
        taken, took = run()
        assert taken and 0.03 < took < 0.2
        fcntl.flock(other, fcntl.LOCK_EX)  # one that does not end: not for ever
        taken, took = run()
        assert not taken and 0.2 < took < 1.0
        for _ in range(4):  # and less long each time
            taken, took = run()
        assert not taken and took < 0.1
    finally:
        os.close(other)
    assert run()[0]
    assert eng.get_resident()[0]
