"""The rule that picks wavefronts per replica, at the edges of its range: the
results are the CPU replay's bits whatever it picks.

Split launches read the KDE points, the pair list, the restraint targets and
the PSP rows through the caches, keep the pocket in LDS where it fits, and
share an engine with complexes that cannot be split."""
import numpy as np
import pytest

import oracle_lib as O
from gpudock_amd import remc, synth

pytestmark = pytest.mark.gpu

KEYS = ("energy_final", "move_final", "energy_best", "move_best", "acs_mc", "acs_exchg",
        "idx_tmp_final", "step_best", "cmcc_final", "cmcc_best")


def _job(lna, pnp, pnk, n_lig, n_tmp, pos=11, mcc=0, steps=6, spe=3, seed=1):
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=n_lig, n_prt=1, pnk=pnk,
                            pos=pos, seed=seed)
    return remc.JobSpec(cx, remc.temperatures(n_tmp, 0.3, 3.0),
                        remc.mcpara(steps, spe, [0.2] * 3 + [0.05] * 3),
                        remc.default_options(seed=seed, mcc=mcc))


def _same(job, got):
    want = O.replay_run(job.cx, job.temps, job.mc, job.opt)
    for k in KEYS:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize("lna,pnp,pnk,n_lig,n_tmp,pos,mcc,split", [
    (1, 1, 0, 1, 1, 0, 0, 16),           # one replica, one pair
    (17, 65, 64, 2, 8, 64, 1, 16),       # restraints fill the area's slots
    (33, 1037, 1037, 33, 8, 11, 0, 8),   # 264 replicas: more than CUs, two workgroups a CU
    (65, 4000, 3000, 1, 3, 11, 1, 16),   # one workgroup's tables fill the CU's LDS
    (9, 7000, 100, 1, 2, 3, 0, 16),      # pocket read through the caches
    (16, 130, 100, 2, 2, 65, 0, 1)])     # more restraints than the area's slots
def test_split_by_rule(lna, pnp, pnk, n_lig, n_tmp, pos, mcc, split):
    job = _job(lna, pnp, pnk, n_lig, n_tmp, pos, mcc)
    res, rep = remc.batch_run([job])
    assert rep["layout"]["split"] == split
    _same(job, res[0])


def test_split_and_whole_complexes_share_an_engine():
    """One complex that cannot be split no longer keeps the others whole."""
    jobs = [_job(16, 130, 100, 2, 2, pos=65), _job(24, 300, 300, 2, 4, seed=2),
            _job(100, 4000, 500, 1, 2, seed=3)]
    for cfg in ({}, dict(kde_policy=1), dict(persistent=1)):
        res, rep = remc.batch_run(jobs, **cfg)
        assert rep["layout"]["split"] == 16 and rep["layout"]["n_classes"] >= 2
        for job, got in zip(jobs, res):
            _same(job, got)


@pytest.mark.parametrize("split", [8, 4])
@pytest.mark.parametrize("lna,steps,spe", [(3, 6, 3), (24, 12, 4), (61, 68, 34)])
def test_workgroups_of_four_and_eight_share_a_cu(split, lna, steps, spe):
    """Asked for: one replica a workgroup, and two or more workgroups a CU
    (registers for four wavefronts a SIMD; LDS allows two of these complexes'
    or more); fewer atom blocks than wavefronts, and more."""
    job = _job(lna, 200, 200, 2, 4, steps=steps, spe=spe, seed=lna)
    E = remc.Engine(arena_bytes=1 << 26, use_graph=0, split=split)
    h = E.add(job)
    E.cycles(steps // spe)
    E.sync()
    got, _ = E.results(h)
    _same(job, got)
    layout = E.layout()
    assert layout["split"] == split and layout["resident_groups"] >= 2 * 256
    E.close()
