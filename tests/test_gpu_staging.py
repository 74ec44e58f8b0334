"""Transfers of pageable host arrays: states whose size lies just below and
above the lines of the staged path (2 MiB to enter it, pieces of 8 MiB, three
buffers) come back bit for bit, through the state calls and a snapshot."""
import numpy as np
import pytest

from fall3d_amd import ads

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _grid(nbytes, kind, above):
    """A one-bin grid of 8 levels and 12 cells in x whose state has the first
    size at or above (else the last below) nbytes that ny can give."""
    row = 16 * 12 * kind
    ny = -(-nbytes // row) if above else (nbytes - 1) // row
    return 12, ny - 4, 8


@pytest.mark.parametrize("kind,state", [(4, "fp32"), (8, "fp64")])
@pytest.mark.parametrize("above", [False, True])
@pytest.mark.parametrize("mib", [2, 8, 24, 40])
def test_states_come_back(kind, state, mib, above):
    nx, ny, nz = _grid(mib * MIB, kind, above)
    print(f"case: staging {mib} MiB kind {kind} ny {ny}", flush=True)
    a = ads.ADS(nx, ny, nz, 1, "minmod", "rk", kind, state)
    rng = np.random.default_rng(mib + kind)
    c = np.asfortranarray(rng.random(a.shape_c).astype(a.dtype))
    acum = np.asfortranarray(rng.random(a.shape_acum).astype(a.dtype))
    assert (c.nbytes >= mib * MIB) == above
    a.set_state(c, acum)
    for _ in range(2):
        c1, acum1 = a.get_state()
        assert np.array_equal(c1, c) and np.array_equal(acum1, acum)
    blob = a.snapshot(0.0, 0)
    a.set_state(None)
    a.restore(blob)
    c1, acum1 = a.get_state()
    assert np.array_equal(c1, c) and np.array_equal(acum1, acum)
    a.release()
