"""The FP64 pushes' LDS windows and their run tables where they can go wrong:
windows as wide as the grid, runs that pass into the next row or layer, sparse
species (cut runs), particles of exact L, and a current read after moves that
leave the window: a context that re-sorts (run tables, carried re-sorts)
against one that never sorts (plain slices)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,counts,drift", [
    ((3, 2, 5), (700, 0), 0.0),              # every axis inside one window
    ((130, 3, 2), (5000, 40), 0.1),          # rows longer than a wave
    ((17, 13, 11), (60000, 900), 0.4),       # cut runs of a sparse species
    ((33, 31, 8), (1030, 1023), 1.3),        # one particle past a block; fast
    ((64, 64, 9), (90, 0), 0.3),             # most patches and run entries empty
])
@pytest.mark.parametrize("em", [False, True])
def test_pushes_after_a_sort_equal_unsorted_ones(n, counts, drift, em):
    from ctca_amd import emg
    rng = np.random.default_rng(sum(n) + sum(counts))
    total = sum(counts)
    rec = np.zeros(total, dtype=emg.PARTICLE)
    for c, name in enumerate("xyz"):
        rec[name] = rng.random(total) * n[c]
    rec["x"][:2] = [n[0], 0.0]
    rec["y"][:2] = [0.0, n[1]]
    for name in ("vx", "vy", "vz"):
        rec[name] = rng.normal(size=total) * 0.05
    rec["vx"] += drift / 2
    rec["pid"] = np.arange(total)
    q, qm = [0.5, -0.25], [1.0, -0.1]
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))
    core = rng.normal(size=(n[2], n[1], n[0], 6)) * 0.01
    at = [np.arange(-1, v + 2) % v for v in n]
    eb[...] = core[np.ix_(at[2], at[1], at[0])]
    kw = dict(precision=emg.PLAIN_FP64)
    with emg.Context(n, q, qm, [1.0, 1.0], counts, sort_every=3, **kw) as a, \
            emg.Context(n, q, qm, [1.0, 1.0], counts, **kw) as b:
        for ctx in (a, b):
            ctx.upload(rec, counts)
            ctx.set_fields(eb)
        for step in range(5):      # a sort before steps 0 and 3; b never sorts
            for ctx in (a, b):
                ctx.push_em(2) if em else ctx.push_es(2)
            if em:
                # the same FP64 terms, rounded at 2^-49 in the windows
                ja, jb = a.current(), b.current()
                assert np.abs(ja - jb).max() <= 1e-12 * max(1.0, np.abs(jb).max())
            a.deposit_rho(2)
            b.deposit_rho(2)
            for s in range(2):
                ra, rb = a.rho(species=s), b.rho(species=s)
                assert np.abs(ra - rb).max() <= 1e-12 * max(1.0, np.abs(rb).max())
                assert ra.sum() == pytest.approx(q[s] * counts[s], rel=1e-11, abs=1e-11)
        pa, _ = a.download()
        pb, _ = b.download()
    back = np.empty_like(pa)
    back[pa["pid"]] = pa
    assert np.array_equal(back, pb)    # a sort permutes, nothing else
