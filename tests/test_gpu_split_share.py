"""Split workgroups that several replicas share, at the edges of the sharing:
the results are the CPU replay's bits for one to four replicas a workgroup, a
ragged last workgroup, cycles longer than one batch of draws, pockets on both
sides of the two-chunk loop, and every option that a step's end looks at."""
import numpy as np
import pytest

import oracle_lib as O
from gpudock_amd import remc, synth

pytestmark = pytest.mark.gpu

KEYS = ("energy_final", "move_final", "energy_best", "move_best", "acs_mc", "acs_exchg",
        "idx_tmp_final", "step_best", "cmcc_final", "cmcc_best")


@pytest.mark.parametrize("lna,pnp,pnk,n_lig,n_prt,n_tmp,pos,steps,spe,split,opt", [
    (5, 60, 40, 75, 1, 8, 3, 4, 2, 0, {}),                    # 600 replicas: three a workgroup
    (17, 700, 300, 113, 1, 8, 11, 2, 2, 0, dict(mcc=1)),      # 904: four
    (15, 770, 0, 41, 1, 7, 0, 2, 1, 0, dict(combine=1)),      # 287: two, ragged, no KDE
    (4, 64, 30, 91, 1, 3, 2, 66, 33, 0, {}),                  # two batches of draws a cycle
    (5, 130, 40, 5, 2, 33, 5, 4, 2, 4, dict(term_order=1)),   # asked for: four
    (14, 704, 100, 3, 1, 2, 64, 9, 3, 16, dict(term_order=1, reverse=1)),
    (128, 833, 2000, 2, 1, 2, 11, 6, 3, 4, dict(away=1)),     # workgroups of four wavefronts
    (2, 64, 1, 1, 1, 3, 1, 40, 40, 8, dict(fixed_draws=1)),   # of eight
])
def test_shared_workgroups(lna, pnp, pnk, n_lig, n_prt, n_tmp, pos, steps, spe, split, opt):
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=n_lig, n_prt=n_prt, pnk=pnk,
                            pos=pos, seed=lna)
    job = remc.JobSpec(cx, remc.temperatures(n_tmp, 0.3, 3.0),
                       remc.mcpara(steps, spe, [0.2] * 3 + [0.05] * 3),
                       remc.default_options(seed=lna, **opt))
    want = O.replay_run(job.cx, job.temps, job.mc, job.opt)
    for persistent in (0, 1):
        res, rep = remc.batch_run([job], split=split, persistent=persistent)
        n_rep = n_lig * n_prt * n_tmp
        by_rule = 16 // -(-n_rep // 256)
        assert rep["layout"]["split"] == (split or by_rule)
        for k in KEYS:
            np.testing.assert_array_equal(res[0][k], want[k], err_msg=k)


@pytest.mark.parametrize("lna,pnp,n_tmp", [(9, 100, 2), (100, 4000, 2)])
def test_autotune_tries_every_sharing(lna, pnp, n_tmp):
    """Also where the tables leave room for one area only."""
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=2, n_prt=1, pnk=60, pos=2,
                            seed=lna)
    job = remc.JobSpec(cx, remc.temperatures(n_tmp, 0.3, 3.0),
                       remc.mcpara(4, 2, [0.2] * 3 + [0.05] * 3), remc.default_options(seed=1))
    res, rep = remc.batch_run([job], autotune=1)
    assert rep["tune"]["n"] > 6
    want = O.replay_run(job.cx, job.temps, job.mc, job.opt)
    for k in KEYS:
        np.testing.assert_array_equal(res[0][k], want[k], err_msg=k)
