"""The FP64 zigzag current of particles that cross several cells in a step: the
relay point of such a move lies at the far cell (or at the box face), so its
weights are not within [0, 1]."""
import numpy as np
import pytest

import oracle
from ctca_amd import emg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["slices", "patches", "rows"])
@pytest.mark.parametrize("ustep", [1, 2])
@pytest.mark.parametrize("axes", [1, 2, 3])
@pytest.mark.parametrize("cells", [2, 3, 4, 6, 8])
def test_current_of_moves_over_several_cells(cells, axes, ustep, order):
    n = (24, 20, 18)
    counts = (3000, 700)
    q, qm, rm = (0.5, -0.25), (1.0, -0.1), (1.0, 1.0)
    rng = np.random.default_rng(100 * cells + 10 * axes + ustep)
    total = sum(counts)
    p = np.zeros(total, dtype=emg.PARTICLE)
    for c, name in enumerate("xyz"):
        p[name] = rng.random(total) * n[c]
    for c, name in enumerate(("vx", "vy", "vz")):
        move = rng.uniform(-0.5, 0.5, total)
        # the axes rotate over the particles, so that each is a fast one
        fast = (np.arange(total) + c) % 3 < axes
        move[fast] += cells * rng.choice([-1.0, 1.0], total)[fast]
        p[name] = move / ustep
    p["pid"] = np.arange(total)
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))
    core = rng.normal(size=(n[2], n[1], n[0], 6)) * 0.01
    at = [np.arange(-1, v + 2) % v for v in n]
    eb[...] = core[np.ix_(at[2], at[1], at[0])]
    with emg.Context(n, q, qm, rm, counts, precision=emg.PLAIN_FP64,
                     sort_every=1 if order == "patches" else 0) as ctx:
        ctx.upload(p, counts)
        ctx.set_fields(eb)
        if order == "rows":
            ctx.sort()
        ctx.push_em(ustep)
        got = ctx.current(lo=(-1, -1, -1), hi=tuple(v + 1 for v in n))
        g, _ = ctx.download()
    o = p.copy()
    wrk = oracle.grdcrt(eb, n, (0, 0, 0), (0, 0, 0))
    aj = oracle.psolve1(o, counts, qm, q, wrk, n, ustep, np.array(n, dtype=float))
    oracle.fold_current(aj, n)
    want = aj[3:n[2] + 6, 3:n[1] + 6, 3:n[0] + 6]   # indices -1 .. n+1
    g = g[np.argsort(g["pid"], kind="stable")]
    for f in ("x", "y", "z", "vx", "vy", "vz"):
        assert np.array_equal(g[f], o[f]), f
    # a node sums some tens of terms, each rounded at 2^-49 or 2^-53 of the largest
    assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
