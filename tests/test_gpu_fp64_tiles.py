"""The charge of an unsorted FP64 state, binned by tiles: against numpy's CIC on
grids with partial tiles, less than a tile, and more tiles than a workgroup
counts in LDS; particles on the box faces; an empty and a third species; an
ordered upload, which keeps the blocks' windows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cic(rec, n):
    out = np.zeros(n[0] * n[1] * n[2])
    pos = [rec[c] for c in "xyz"]
    i = [np.minimum(p.astype(np.int64), n[d] - 1) for d, p in enumerate(pos)]
    f = [p - c for p, c in zip(pos, i)]
    for q in range(8):
        o = [(q >> d) & 1 for d in range(3)]
        g = [(i[d] + o[d]) % n[d] for d in range(3)]
        w = np.prod([f[d] if o[d] else 1.0 - f[d] for d in range(3)], axis=0)
        out += np.bincount((g[2] * n[1] + g[1]) * n[0] + g[0], w, len(out))
    return out.reshape(n[2], n[1], n[0])


@pytest.mark.parametrize("n,counts,ordered", [
    ((16, 16, 16), (131071, 0, 1), False),        # the smallest that is binned
    ((5, 300, 3), (100000, 50000, 20000), False),
    ((33, 9, 70), (150000, 1, 60000), False),
    ((136, 136, 128), (90000, 60000, 0), False),  # 4,624 tiles
    ((40, 40, 40), (2200000, 30000, 4096), False),  # long slices
    ((40, 40, 40), (140000, 30000, 4096), True),
])
def test_charge_of_an_unsorted_state(n, counts, ordered):
    from ctca_amd import emg
    total = sum(counts)
    rng = np.random.default_rng(total)
    rec = np.zeros(total, dtype=emg.PARTICLE)
    for c, name in enumerate("xyz"):
        rec[name] = rng.random(total) * n[c]
    rec["x"][5:9] = [0.0, n[0], n[0] - 1e-12, 0.5]
    rec["z"][5:9] = [n[2], n[2], 0.0, n[2] - 1.0]
    for name in ("vx", "vy", "vz"):
        rec[name] = rng.normal(size=total) * 0.02
    if ordered:
        off = 0
        for c in counts:
            seg = rec[off:off + c]
            seg[:] = seg[np.lexsort((seg["x"].astype(int), seg["y"].astype(int),
                                     seg["z"].astype(int)))]
            off += c
    q = [0.5, -2.0, 1.0]
    with emg.Context(n, q, [1.0, -1.0, 0.5], [1.0] * 3, counts) as ctx:
        ctx.upload(rec, counts)
        ctx.set_fields(np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6)))
        for moved in (False, True):
            if moved:
                ctx.push_es(2)
            ctx.deposit_rho(2)
            now, _ = ctx.download()
            off = 0
            for s, c in enumerate(counts):
                want = q[s] * _cic(now[off:off + c], n)
                got = ctx.rho(species=s)
                # sums of the same FP64 weights in another order: k terms per node
                k = 8 * (c / (n[0] * n[1] * n[2]) + 8)
                assert np.abs(got - want).max() <= 4 * k * 2.2e-16 * max(np.abs(want).max(), 1.0)
                off += c
        for name in ("x", "y", "z"):     # free streaming of the pushed positions
            d = now[name] - rec[name] - 2.0 * rec["v" + name]
            L = n["xyz".index(name)]
            assert np.abs(d - L * np.round(d / L)).max() <= 1e-12
