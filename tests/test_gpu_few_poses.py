"""Few poses at once: each split over a workgroup's wavefronts, one to four
poses a workgroup.  Energies are the CPU replay's bits at the edges of that
path, and runs without exchange, whose cycles share a launch, end as the
replay's do."""
import numpy as np
import pytest

import oracle_lib as O
from gpudock_amd import remc, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_pose,lna,pnp,pnk,n_lig,n_prt,pos,order", [
    (1, 1, 1, 0, 1, 1, 0, 0),
    (3, 16, 64, 30, 2, 2, 64, 1),
    (257, 17, 65, 500, 3, 1, 1, 0),      # two a workgroup, the last one ragged
    (600, 9, 130, 64, 4, 3, 11, 0),      # three
    (1021, 24, 300, 300, 4, 5, 11, 1),   # four
    (3583, 5, 70, 60, 2, 1, 2, 0),       # the last count that is split
    (3584, 5, 70, 60, 2, 1, 2, 0),       # and the first that is not
    (5, 128, 4000, 5000, 2, 1, 11, 0),   # one fits beside the tables
    (4, 65, 7000, 200, 1, 1, 3, 0),      # pocket read through the caches
    (6, 20, 200, 100, 1, 1, 65, 0)])     # more restraints than the area's slots
@pytest.mark.parametrize("noalloc", [False, True])
def test_few_poses(n_pose, lna, pnp, pnk, n_lig, n_prt, pos, order, noalloc):
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=n_lig, n_prt=n_prt, pnk=pnk,
                            pos=pos, seed=n_pose)
    rng = np.random.default_rng(n_pose)
    lc = rng.integers(0, n_lig, n_pose).astype(np.int32)
    pc = rng.integers(0, n_prt, n_pose).astype(np.int32)
    mv = np.concatenate([rng.normal(0, 0.6, (n_pose, 3)), rng.normal(0, 0.4, (n_pose, 3))], 1)
    e = remc.score_poses(cx, lc, pc, mv.astype(np.float32), term_order=order, fp64=False,
                         noalloc=noalloc)
    np.testing.assert_array_equal(e, O.replay_energy(cx, lc, pc, mv, term_order=order))


@pytest.mark.parametrize("split", [0, 1])
def test_cycles_of_one_launch(split):
    """Different steps, exchange steps and windows in one engine, none with
    temperatures to swap; one job beside them that swaps ends the sharing."""
    def job(i, n_tmp, steps, spe, dump=None, **opt):
        cx = synth.make_complex(pnp=60 + i, radius=None, lna=4 + i, n_lig=2, n_prt=1, pnk=30,
                                pos=2, seed=i)
        return remc.JobSpec(cx, remc.temperatures(n_tmp, 0.3, 3.0),
                            remc.mcpara(steps, spe, [0.2] * 3 + [0.05] * 3, dump),
                            remc.default_options(seed=i, complex_id=i, **opt))
    alone = [job(1, 1, 1700, 7), job(2, 3, 40, 10, exchange=0), job(3, 1, 9, 4, 6)]
    for jobs in (alone, alone + [job(4, 2, 60, 5)]):
        for no_graph in (0, 1):
            res, _ = remc.batch_run(jobs, split=split, no_graph=no_graph)
            for j, got in zip(jobs, res):
                want = O.replay_run(j.cx, j.temps, j.mc, j.opt)
                for k in ("energy_final", "move_final", "energy_best", "acs_mc", "acs_exchg",
                          "idx_tmp_final", "step_best"):
                    np.testing.assert_array_equal(got[k], want[k], err_msg=k)
