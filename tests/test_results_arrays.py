"""The arrays made of a result struct array hold its fields' values."""
import ctypes as C

import numpy as np
import pytest

from gpudock_amd import remc


@pytest.mark.parametrize("n", [0, 1, 65])
def test_results_to_numpy(n):
    res = (remc.ReplicaResult * n)()
    raw = np.random.default_rng(n).integers(0, 60, C.sizeof(res)).astype(np.uint8)
    C.memmove(res, raw.tobytes(), C.sizeof(res))
    out = remc.results_to_numpy(res)
    assert list(out) == ["move_final", "energy_final", "move_best", "energy_best",
                         "energy_best_fp64", "step_best", "idx_tmp_final", "acs_mc",
                         "acs_exchg", "cmcc_final", "cmcc_best"]
    for name, kind in remc.ReplicaResult._fields_:
        width = getattr(kind, "_length_", 0)
        a = out[name]
        assert a.shape == ((n, width) if width else (n,)) and a.flags.c_contiguous
        assert a.dtype == np.dtype(getattr(kind, "_type_", kind) if width else kind)
        want = [list(getattr(r, name)) if width else getattr(r, name) for r in res]
        np.testing.assert_array_equal(a, np.array(want, a.dtype).reshape(a.shape))
    for a in out.values():
        a[...] = 0   # arrays of their own
    assert bytes(res) == raw.tobytes()


def test_results_to_numpy_of_any_sequence():
    """A slice of a result array, a list and a tuple of picked replicas."""
    res = (remc.ReplicaResult * 9)()
    for i, r in enumerate(res):
        r.step_best, r.move_best[2], r.energy_best_fp64[9] = i, 0.5 * i, -1.0 / (i + 1)
    for part, ids in ((res[2:7], range(2, 7)), ([res[8], res[0]], (8, 0)),
                      (tuple(res), range(9)), ([], ())):
        out = remc.results_to_numpy(part)
        np.testing.assert_array_equal(out["step_best"], list(ids))
        np.testing.assert_array_equal(out["move_best"][:, 2], [0.5 * i for i in ids])
        np.testing.assert_array_equal(out["energy_best_fp64"][:, 9], [-1.0 / (i + 1) for i in ids])
        assert out["move_best"].shape == (len(ids), 6)
