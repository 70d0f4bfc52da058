"""Transfers of one context from several threads: the runs of a batch read and
written at once, and a run watched while it steps.  Transfers convert in a
buffer that the steps write too, so a mix-up shows in the values."""
import threading

import numpy as np
import pytest
import torch   # before the library: one HIP runtime in the process

from amun_amd.problems import kelvin_helmholtz_2d
from amun_amd.solver import Batch, Solver
from test_gpu_batch import _kh_runs
from test_gpu_cells import _params, _state

pytestmark = pytest.mark.gpu


def _together(jobs):
    """run the jobs on a thread each; the first exception is raised here"""
    errors = []

    def call(f):
        try:
            f()
        except BaseException as e:      # noqa: BLE001 -- reported below
            errors.append(e)
    threads = [threading.Thread(target=call, args=(f,)) for f in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
        assert not t.is_alive()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_transfers_from_threads(precision):
    common, runs = _kh_runs([64, 128, 32, 96, 64, 160], precision)
    u0 = [kelvin_helmholtz_2d(p, seed=i) for i, p in enumerate(runs)]
    print(f"[case] batch transfers {precision}", flush=True)
    with Batch(common, runs) as a, Batch(common, runs) as b:
        for r, u in enumerate(u0):
            a.upload(r, u)
        _together([lambda r=r: b.upload(r, u0[r]) for r in range(len(runs))])
        np.testing.assert_array_equal(b.run(3), a.run(3))
        want = [a.download(r, with_q=True) for r in range(len(runs))]

        def read(r):
            for _ in range(10):
                u, q = b.download(r, with_q=True)
                np.testing.assert_array_equal(u, want[r][0])
                np.testing.assert_array_equal(q, want[r][1])
        _together([lambda r=r: read(r) for r in range(len(runs))])


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("case", [(2, "mhd", "tvd", 16, (6, 4)), (3, "mhd", "weno5z", 16, (7, 6, 6))])
def test_download_while_stepping(case, graph):
    """The run goes on as if nobody watched, and every download is the state
    after a whole step (the larger state, 71 MiB, comes in staged pieces)."""
    p = _params(*case)
    u0 = _state(p)
    n = 12
    print(f"[case] stepping {case} graph={graph}", flush=True)
    with Solver(p) as s:
        s.upload(u0)
        states, dts = [s.download()], []
        for _ in range(n):
            dts.append(s.run(1)[0])
            states.append(s.download())
    seen = []
    with Solver(p) as s:
        s.set_graph(graph)
        s.upload(u0)

        def watch():
            for _ in range(4):
                seen.append(s.download())
        got = []
        _together([lambda: got.append(s.run(n)), watch])
        np.testing.assert_array_equal(got[0], dts)
        np.testing.assert_array_equal(s.download(), states[-1])
    for u in seen:
        assert any(np.array_equal(u, v) for v in states)


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two devices")
def test_large_download_from_a_thread_on_another_device():
    p = _params(3, "mhd", "weno5z", 16, (7, 6, 6))
    u0 = _state(p)
    print("[case] download on another device's thread", flush=True)
    with torch.cuda.device(1), Solver(p) as s:
        s.upload(u0)
        got = []
        _together([lambda: got.extend(s.download() for _ in range(2))])
        for u in got:
            np.testing.assert_array_equal(u, u0)
        assert torch.cuda.current_device() == 1
