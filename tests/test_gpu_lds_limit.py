"""The kernels' dynamic LDS limit is the process's, not a call's: an engine
whose tables fill a CU's LDS goes on after calls on a small complex, between
its cycles and from another thread."""
import ctypes as C
import re
import subprocess
import threading

import numpy as np
import pytest

import oracle_lib as O
from gpudock_amd import remc, synth

pytestmark = pytest.mark.gpu

KEYS = ("energy_final", "move_final", "energy_best", "acs_mc", "acs_exchg", "step_best")


def _big():
    cx = synth.make_complex(pnp=4000, radius=None, lna=20, n_lig=2, n_prt=1, pnk=300, pos=2, seed=4)
    return remc.JobSpec(cx, remc.temperatures(4, 0.3, 3.0),
                        remc.mcpara(24, 2, [0.2] * 3 + [0.05] * 3), remc.default_options(seed=4))


def _score_small(n):
    cx = synth.make_complex(pnp=64, radius=None, lna=5, n_lig=1, n_prt=1, pnk=10, pos=1, seed=n)
    z = np.zeros(n, np.int32)
    mv = np.random.default_rng(n).normal(0, 0.5, (n, 6)).astype(np.float32)
    e = remc.score_poses(cx, z, z, mv, fp64=False)
    np.testing.assert_array_equal(e, O.replay_energy(cx, z, z, mv))


@pytest.mark.parametrize("split", [1, 0])
def test_small_calls_between_the_cycles_of_a_large_engine(split):
    job = _big()
    E = remc.Engine(arena_bytes=1 << 28, use_graph=0, split=split)
    h = E.add(job)
    for n in (1, 4000, 3):
        E.cycles(4)
        E.sync()
        assert E.layout()["stage_bytes"] > 90000
        _score_small(n)
    got, _ = E.results(h)
    want = O.replay_run(job.cx, job.temps, job.mc, job.opt)
    for k in KEYS:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    E.close()


class _FuncAttributes(C.Structure):   # hipFuncAttributes
    _fields_ = [("binary_version", C.c_int), ("cache_mode", C.c_int), ("const_bytes", C.c_size_t),
                ("local_bytes", C.c_size_t), ("max_dynamic", C.c_int), ("max_threads", C.c_int),
                ("num_regs", C.c_int), ("carveout", C.c_int), ("ptx_version", C.c_int),
                ("shared_bytes", C.c_size_t)]


def test_a_small_call_leaves_every_kernels_limit_alone():
    lib = remc.lib()
    hip = C.CDLL("libamdhip64.so")
    _score_small(2)
    names = subprocess.run(["nm", "-D", "--defined-only", lib._name], check=True,
                           capture_output=True, text=True).stdout.split()
    names = [n for n in names if re.match(r"_Z\d+gd_(mc|mc_split|score|pose_split|rescore64)_kernel", n)]
    assert len(names) > 3
    for n in names:
        a = _FuncAttributes()
        assert hip.hipFuncGetAttributes(C.byref(a), C.c_void_p(C.addressof(
            C.c_char.in_dll(lib, n)))) == 0, n
        assert a.max_dynamic >= 160 * 1024 - 64, n


def test_large_and_small_calls_from_two_threads():
    job = _big()
    want = O.replay_run(job.cx, job.temps, job.mc, job.opt)
    stop, errors = threading.Event(), []

    def small():
        try:
            while not stop.is_set():
                _score_small(2)
        except Exception as e:   # noqa: BLE001 -- handed to the test's thread
            errors.append(e)

    t = threading.Thread(target=small)
    t.start()
    try:
        for _ in range(10):
            got, _ = remc.run(job.cx, job.temps, job.mc, job.opt)
            for k in KEYS:
                np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    finally:
        stop.set()
        t.join()
    assert not errors, errors[0]
