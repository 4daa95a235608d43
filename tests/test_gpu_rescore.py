"""The FP64 re-score kernel at the edges of its work split, against the FP64
oracle and against itself.

A pose's atoms, KDE rounds and restraints are summed in eight slices, by
eight wavefronts or by four, so the sizes around multiples of 8 atoms and 64
points are tried, and pose counts on both sides of the rule that picks the
wavefronts (four poses a CU: 1,024).  Tolerance: a pair term is formed by
about 15 roundings of 2^-53, 1.7e-15 of the term; the signed sums cancel at
most three decimal digits of the terms' magnitude here, and the weights are
below 10: 2e-11 of max(|E|, 1) bounds every slot."""
import numpy as np
import pytest

import oracle_lib as O
from gpudock_amd import remc, synth

pytestmark = pytest.mark.gpu

TOL = 2e-11


def _poses(seed, n, n_lig, n_prt):
    rng = np.random.default_rng(seed)
    lc = rng.integers(0, n_lig, n).astype(np.int32)
    pc = rng.integers(0, n_prt, n).astype(np.int32)
    mv = np.concatenate([rng.normal(0, 0.5, (n, 3)), rng.normal(0, 0.5, (n, 3))], 1)
    return lc, pc, mv.astype(np.float32)


@pytest.mark.parametrize("lna,pnp,pnk,pos", [
    (1, 1, 0, 0), (7, 64, 40, 7), (8, 65, 64, 8), (9, 127, 700, 9), (16, 128, 0, 11),
    (17, 300, 300, 1), (64, 129, 1600, 17), (65, 200, 1600, 0), (128, 190, 3000, 11),
    (40, 6000, 200, 3)])
def test_fp64_slices_against_the_oracle(lna, pnp, pnk, pos):
    """The last size's pocket does not fit LDS beside the table."""
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=3, n_prt=2, pnk=pnk, pos=pos,
                            seed=100 + lna)
    lc, pc, mv = _poses(lna, 13, 3, 2)
    for order in (remc.TERM_ORDER_FILE, remc.TERM_ORDER_SLOT):
        _, e64 = remc.score_poses(cx, lc, pc, mv, term_order=order)
        r64 = O.pose_ref64(cx, lc, pc, mv, term_order=order)
        np.testing.assert_allclose(e64, r64, rtol=TOL, atol=TOL)


def test_fp64_same_bits_whatever_shares_the_launch():
    """Eight wavefronts per pose up to 1,024 poses, four beyond."""
    cx = synth.make_config("c0", n_lig=3, n_prt=2)[0]
    lc, pc, mv = _poses(5, 1025, 3, 2)
    _, many = remc.score_poses(cx, lc, pc, mv)
    _, few = remc.score_poses(cx, lc[:1024], pc[:1024], mv[:1024])
    _, one = remc.score_poses(cx, lc[700:701], pc[700:701], mv[700:701])
    np.testing.assert_array_equal(many[:1024], few)
    np.testing.assert_array_equal(many[700:701], one)


def test_fp64_degenerate_distances():
    """An atom on a pocket point and an infinite translation: the soft-LJ
    quotient has no value there, every other term has the oracle's."""
    cx = synth.make_config("c0", n_lig=1, n_prt=1)[0]
    cx.prt_xyz[0, 17] = cx.lig_xyz[0, 5] + cx.lig_center
    cx._build()
    mv = np.zeros((2, 6), np.float32)
    mv[1, 1] = np.inf
    z = np.zeros(2, np.int32)
    _, e64 = remc.score_poses(cx, z, z, mv)
    with np.errstate(all="ignore"):
        r64 = O.pose_ref64(cx, z, z, mv)
    vdw = remc.SLOTS.index("vdw")
    assert np.isnan(r64[:, vdw]).all() and np.isfinite(r64[0, 1:9]).all()
    np.testing.assert_allclose(e64, r64, rtol=TOL, atol=TOL)


@pytest.mark.parametrize("lna,pnp,pnk,pos", [(24, 300, 300, 11), (65, 129, 700, 0)])
def test_fp64_nan_poses_keep_their_nan(lna, pnp, pnk, pos):
    """A NaN of either sign in the translation or an angle, and an infinite
    angle: every term that the oracle gives as NaN is NaN, the others have its
    value, and the poses beside them are untouched."""
    cx = synth.make_complex(pnp=pnp, radius=None, lna=lna, n_lig=1, n_prt=1, pnk=pnk, pos=pos,
                            seed=lna)
    mv = np.zeros((8, 6), np.float32)
    mv[1, 0] = np.nan
    mv[2, 2] = -np.float32(np.nan)
    mv[3, 4] = np.nan
    mv[4, 3] = np.inf
    mv[6, :] = np.nan
    z = np.zeros(len(mv), np.int32)
    with np.errstate(all="ignore"):
        r64 = O.pose_ref64(cx, z, z, mv)
    for name in ("hdb", "kde"):
        k = remc.SLOTS.index(name)
        assert np.isnan(r64[[1, 2, 3, 4, 6], k]).all() and np.isfinite(r64[[0, 5, 7], k]).all()
    for noalloc in (False, True):
        _, e64 = remc.score_poses(cx, z, z, mv, noalloc=noalloc)
        np.testing.assert_allclose(e64, r64, rtol=TOL, atol=TOL)
