"""Gram-Schmidt with one launch per state (k_gs_state) against the FP64 oracle
at the edges of its tiles and layouts: ranks around the 16-row tiles, basis
sizes around the 16-column tiles and the two-column slices, one to many modes,
blocks with more states than the device has room for workgroups, and the
kernel-per-step form it falls back to.

Tolerance as in the other parity tests: represented tensors 1e-9 relative
(rounding amplified by a few ALS sweeps)."""
import sys

import numpy as np
import pytest

from tests.helpers import full_tensor, random_block, random_system

pytestmark = pytest.mark.gpu

TOL_T = 1e-9

CASES = [
    ("tile1", [15, 16, 17], [1, 15, 16, 3]),
    ("tile2", [16, 33, 9], [17, 31, 32, 8, 18]),
    ("tile3", [20, 47, 18], [33, 47, 48, 16]),
    ("tile4", [24, 31, 32], [49, 63, 64, 17]),
    ("slice", [64, 12, 8], [5, 20, 7]),
    ("slices2", [65, 9, 10], [6, 19, 33]),
    ("widest", [128, 7, 97], [9, 40, 64]),
    ("unit", [1, 2, 1, 3], [1, 2, 1]),
    ("five", [4, 6, 3, 5, 4], [7, 2, 9, 5]),
    ("onemode", [9], [1, 1, 1, 1]),
]


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


def ortho(Q, H, nals, form=None):
    from mlcp_amd.intertwine import Session
    with Session(Q, H) as s:
        if form:
            s.set_form(*form)
        s.ortho(nals)
        return s.download(), s.sweeps()[0].copy()


def tensors(Q):
    return [full_tensor(Q.nbas, *Q.state(s)) for s in range(Q.nbloc)]


@pytest.mark.parametrize("name,nb,ranks", CASES)
def test_states_against_oracle(hip, name, nb, ranks):
    from oracle.orc import C
    say("states", name, nb, ranks)
    H = random_system(3, nb, ncoup=2 if len(nb) > 1 else 0)
    Q = random_block(4, nb, ranks)
    g, _ = ortho(Q, H, 3)
    o = C.als_ortho3(Q, 3)
    for a, b in zip(tensors(g), tensors(o)):
        assert np.linalg.norm(a - b) < TOL_T * np.linalg.norm(b)


def test_more_states_than_workgroups(hip):
    """240 states: the last ones run kernel by kernel behind the others."""
    from oracle.orc import C
    nb, ranks = [65, 66], [2] * 240
    say("many states", nb, len(ranks))
    H = random_system(5, nb, ncoup=1)
    Q = random_block(6, nb, ranks)
    g, _ = ortho(Q, H, 2)
    o = C.als_ortho3(Q, 2)
    for s in range(0, 240, 13):
        a, b = (full_tensor(x.nbas, *x.state(s)) for x in (g, o))
        assert np.linalg.norm(a - b) < TOL_T * np.linalg.norm(b), s


def test_wait_that_runs_out_is_run_again(hip, monkeypatch):
    """One poll per wait: the hand-overs give up, every workgroup leaves, and
    the call returns what the kernel-per-step form gives, bit for bit."""
    from mlcp_amd.intertwine import Session
    nb, ranks = [12, 9, 14], [18, 7, 33, 12]
    H, Q = random_system(7, nb, ncoup=3), random_block(8, nb, ranks)
    say("retry", nb, ranks)
    monkeypatch.setenv("MLCP_HIP_GS_SPIN", "0")
    with Session(Q, H) as s:
        e0 = s.cycle(np.zeros(4), 1, 3, True, 1, 4.0)
        g0 = s.download()
    monkeypatch.setenv("MLCP_HIP_GS_SPIN", "1")
    with Session(Q, H) as s:
        e1 = s.cycle(np.zeros(4), 1, 3, True, 1, 4.0)
        g1 = s.download()
        e2 = s.cycle(np.zeros(4), 1, 3, True, 1, 4.0)
    assert np.array_equal(e0, e1) and np.all(np.isfinite(e2))
    assert np.array_equal(g0.base, g1.base) and np.array_equal(g0.coef, g1.coef)


def test_tolerance_form_stops_at_the_same_sweeps(hip, monkeypatch):
    nb, ranks = [14, 11, 9], [6, 17, 9, 12]
    H, Q = random_system(9, nb, ncoup=3), random_block(10, nb, ranks)
    say("tolerance", nb, ranks)
    out = {}
    for spin in ("0", "1000000"):
        monkeypatch.setenv("MLCP_HIP_GS_SPIN", spin)
        out[spin] = ortho(Q, H, 8, (1, 1e-3, 1e-7))
    (a, sa), (b, sb) = out.values()
    assert np.array_equal(sa, sb) and sa.max() > 0
    for x, y in zip(tensors(a), tensors(b)):
        assert np.linalg.norm(x - y) < TOL_T * np.linalg.norm(y)
