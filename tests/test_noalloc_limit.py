"""The largest call that gd_score_poses_noalloc takes: what counts against the
static workspace alone decides, in FP32 and with FP64 energies, for one
protein conformer and for several.  Checked before any device work, so it
runs without a GPU too (an accepted call then ends with "no HIP device")."""
import re

import numpy as np
import pytest

from gpudock_amd import remc, synth

LIMIT = 64 << 20


def _refused(cx, n, n_prt):
    """None when the call is taken, else the bytes it is said to need."""
    zeros = np.zeros(n, np.int32)
    prt = (np.arange(n) % n_prt).astype(np.int32)
    mv = np.zeros((n, 6), np.float32)
    e = np.zeros((n, 10), np.float32)
    e64 = np.zeros((n, 10), np.float64)
    rc = remc.lib().gd_score_poses_noalloc(
        *cx.args(), cx.size, n, remc._ip(zeros), remc._ip(prt), remc._fp(mv), 0, 0, remc._fp(e),
        e64.ctypes.data_as(remc.C.POINTER(remc.C.c_double)))
    if rc == 0:
        return None
    text = remc.lib().gd_last_error().decode()
    if "static workspace" not in text and "gd_score_poses_noalloc" not in text:
        assert "no HIP device" in text, text
        return None
    found = re.search(r"need (\d+) bytes", text)
    assert found, text
    return int(found.group(1))


@pytest.mark.parametrize("n_prt", [1, 7])
def test_largest_call_with_fp64(n_prt):
    cx = synth.make_complex(pnp=300, radius=None, lna=24, n_lig=1, n_prt=n_prt, pnk=300, pos=11,
                            seed=n_prt)
    lo, hi = 300000, 500000
    assert _refused(cx, lo, n_prt) is None and _refused(cx, hi, n_prt) > LIMIT
    while hi - lo > 1:
        mid = (lo + hi) // 2
        if _refused(cx, mid, n_prt) is None:
            lo = mid
        else:
            hi = mid
    # one pose more is 158 bytes, with every array rounded up to 256
    assert LIMIT < _refused(cx, hi, n_prt) <= LIMIT + 7 * 256 + 158
