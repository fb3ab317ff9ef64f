"""Host transfers of any size: states below and above the size that passes through the pinned slots, with
remainders of a slot, from several threads at once, come back as they went."""
import ctypes as C
import sys
import threading

import numpy as np
import pytest

from flowmol_amd import config
from flowmol_amd._lib import check, load
from flowmol_amd.md import MDContext

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def round_trip(n, seed, times, failed):
    try:
        rng = np.random.default_rng(seed)
        p = config.make_params((60.0, 60.0, 60.0), n / 60.0 ** 3, 2.5)
        g = None
        for _ in range(times):
            r, v, a = (rng.uniform(-29.0, 29.0, (n, 3)) for _ in range(3))
            if g is None:
                g = MDContext(p, r, v, a)
            else:
                g.upload_state(r, v, a)
            for sent, got in zip((r, v, a), g.state()):
                assert np.array_equal(sent, got)
        g.close()
    except Exception as e:  # noqa: BLE001 (reported by the caller)
        failed.append(e)


# 72 bytes a molecule: 4 MiB is 58,254 of them, a 2 MiB slot 87,381 vectors
@pytest.mark.parametrize("n", [1, 58254, 58255, 87381, 87382, 300001])
def test_round_trip(n):
    say(f"case: {n} molecules up and down")
    failed = []
    round_trip(n, n, 2, failed)
    assert not failed, failed


def test_round_trips_from_seven_threads():
    say("case: seven threads, a context each, 70,000 molecules")
    failed = []
    th = [threading.Thread(target=round_trip, args=(70000 + k, k, 3, failed)) for k in range(7)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not failed, failed


def placed(x, where):
    """A copy of x in the named kind of memory, with the object that keeps it and its address."""
    import torch

    t = torch.from_numpy(np.ascontiguousarray(x))
    t = {"pinned": lambda: t.pin_memory(), "device": lambda: t.cuda(), "plain": lambda: t.clone()}[where]()
    torch.cuda.synchronize()
    return t, C.cast(t.data_ptr(), C.POINTER(C.c_double))


@pytest.mark.parametrize("where", [("pinned",) * 3, ("device",) * 3, ("plain", "pinned", "device"),
                                   ("pinned", "plain", "plain")])
def test_arrays_that_the_runtime_knows(where):
    """Pinned and device memory is copied by the device itself, whatever its size, beside plain arrays of
    the same call."""
    p, r, v = config.config_fcc((50, 50, 50), 0.8, 2.5, seed=8, tplot=10)   # 12 MB an array
    rng = np.random.default_rng(8)
    src = [rng.uniform(-1.0, 1.0, r.shape) for _ in range(3)]
    say(f"case: 500000 molecules, arrays {where}")
    g = MDContext(p, r, v)
    given = [placed(x, w) for x, w in zip(src, where)]
    got = [placed(np.zeros_like(x), w) for x, w in zip(src, where)]
    check(load().fm_upload_state(g._h, r.shape[0], *[a for _, a in given]))
    check(load().fm_download_state(g._h, *[a for _, a in got]))
    for x, (t, _) in zip(src, got):
        assert np.array_equal(t.cpu().numpy(), x)
    g.close()


# 8 MiB an array (349,525 molecules) is where slots of one unit (2 MiB) become slots of two and where uploads
# begin to pass through them
@pytest.mark.parametrize("n", [174762, 174763, 349525, 349526, 1100001])
def test_round_trip_at_the_slot_sizes(n):
    say(f"case: {n} molecules up and down, twice")
    failed = []
    round_trip(n, n, 2, failed)
    assert not failed, failed
