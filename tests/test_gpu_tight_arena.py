"""Engines whose arena holds little beside the complexes: one wavefront-sized
task list, 88 bytes a replica for the results, and no more.  Split replicas
have longer task lists and the FP64 re-score its own; both make do with that
room, and the results are the CPU replay's bits."""
import numpy as np
import pytest

import oracle_lib as O
from gpudock_amd import remc, synth

pytestmark = pytest.mark.gpu

KEYS = ("energy_final", "move_final", "energy_best", "move_best", "acs_mc", "acs_exchg",
        "idx_tmp_final", "step_best")


def _job(lna, pnp, pnk, n_lig, n_prt, n_tmp, pos=3, seed=1, **opt):
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=n_lig, n_prt=n_prt, pnk=pnk,
                            pos=pos, seed=seed)
    return remc.JobSpec(cx, remc.temperatures(n_tmp, 0.3, 3.0),
                        remc.mcpara(4, 2, [0.2] * 3 + [0.05] * 3),
                        remc.default_options(seed=seed, **opt))


def _up(n):
    return (n + 255) & ~255


def _room(jobs):
    """Control block, packs, task lists (16 bytes a task: one replica up to 512
    in all, else eight), chains, then 8 + 80 bytes a replica."""
    n = sum(j.n_rep for j in jobs)
    tasks = n if n <= 512 else sum(j.size.n_prt * -(-j.n_rep // j.size.n_prt // 8) for j in jobs)
    chains = sum(j.size.n_prt * j.size.n_lig for j in jobs)
    return (256 + 1024 * len(jobs) + _up(16 * tasks) + _up(8 * chains) + _up(8 * n) + _up(80 * n))


@pytest.mark.parametrize("jobs", [
    [(7, 300, 30, 4, 2, 8)],                                  # 64 replicas
    [(9, 4000, 30, 64, 1, 16)],                               # 1,024, one a split workgroup
    [(5, 1037, 100, 37, 1, 16)],                              # 592, three
    [(4, 800, 50, 37, 3, 8)],                                 # 888, several conformers
    [(3, 70, 10, 33, 1, 31), (8, 3000, 20, 1, 1, 7)],         # 1,030: re-score of two poses
    [(3, 60, 10, 1, 999, 1), (6, 100, 0, 1, 1, 2)],           # one replica a conformer
])
def test_results_in_a_tight_arena(jobs):
    jobs = [_job(*a, seed=i + 2, away=i) for i, a in enumerate(jobs)]
    want = [O.replay_run(j.cx, j.temps, j.mc, j.opt) for j in jobs]
    E = remc.Engine(arena_bytes=sum(_up(j.footprint()) for j in jobs) + _room(jobs), use_graph=0)
    handles = [E.add(j) for j in jobs]
    E.cycles(2)
    E.sync()
    for h, w in zip(handles, want):
        got, _ = E.results(h)
        for k in KEYS:
            np.testing.assert_array_equal(got[k], w[k], err_msg=k)
    E.close()
