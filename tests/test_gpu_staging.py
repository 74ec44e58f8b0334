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


def _address_space():
    for line in open("/proc/self/status"):
        if line.startswith("VmSize:"):
            return int(line.split()[1]) * 1024
    return 0


def test_contexts_share_the_page_locked_buffers():
    """32 contexts (the members of an ensemble) move one large array each: what
    they keep for it does not grow by a set of buffers per context (24 MiB;
    their own transfer area and the allocator's rounding are about 12)."""
    members = [ads.ADS(64, 400, 16, 1, "minmod", "rk", 4, "fp32") for _ in range(32)]
    c = np.zeros(members[0].shape_c, dtype=np.float32, order="F")
    assert c.nbytes >= 2 * MIB
    before = _address_space()
    for g in members:
        g.set_state(c)
    for g in members:
        assert not g.get_state()[0].any()
    grown = _address_space() - before
    print(f"grown {grown / MIB:.0f} MiB", flush=True)
    for g in members:
        g.release()
    assert grown < 32 * 24 * MIB


def test_threads_transfer_side_by_side():
    """Six threads, a context each, more than the buffer sets that wait: every
    state comes back bit for bit."""
    import threading

    errors = []

    def work(k):
        try:
            g = ads.ADS(200, 150, 20 + k, 2, "minmod", "rk", 4, "fp32")
            rng = np.random.default_rng(k)
            for _ in range(3):
                c = np.asfortranarray(rng.random(g.shape_c, dtype=np.float32))
                g.set_state(c)
                if not np.array_equal(g.get_state()[0], c):
                    errors.append(k)
            g.release()
        except Exception as e:  # reported by the test's thread
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
