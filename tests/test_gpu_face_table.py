"""The raw upper-face charge behind the ghost planes, summed per block in an LDS
table: against the oracle, with more nodes than the table holds, with one, and
with most blocks holding none."""
import numpy as np
import pytest

import oracle
from ctca_amd import emg

pytestmark = pytest.mark.gpu


def _fixed_weights(p, n):
    """The FP32 form's raw deposit: each particle's 24-bit weights, which sum to
    2^24, as whole numbers on the nodes -1..n+1."""
    one = np.float32(1)
    cell, f = [], []
    for d, m in zip("xyz", n):
        c = np.floor(p[d])
        o = (p[d] - c).astype(np.float32)
        c = np.where(o >= 1, c + 1, c)
        o = np.where(o >= 1, np.float32(0), o)
        cell.append(c.astype(np.int64) % m)
        f.append(o)
    z = (one - f[2]) * np.float32(2**24), f[2] * np.float32(2**24)
    zy = [(one - f[1]) * z[0], f[1] * z[0], (one - f[1]) * z[1], f[1] * z[1]]
    w = [(a * b).astype(np.int64) for b in zy for a in (one - f[0], f[0])]
    w[7] = 2**24 - sum(w[:7])
    out = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3), dtype=np.int64)
    for k in range(8):
        np.add.at(out, (cell[2] + 1 + (k >> 2), cell[1] + 1 + ((k >> 1) & 1),
                        cell[0] + 1 + (k & 1)), w[k])
    return out.astype(np.float64)


@pytest.mark.parametrize("precision", [emg.PLAIN_FP64, emg.FP32_FIXED], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n,where,counts", [
    ((60, 50, 40), "faces", (40000, 5000)),   # most of a block's nodes are distinct
    ((60, 50, 40), "corner", (3000, 1)),
    ((24, 20, 16), "all", (30000, 1025)),
    ((8, 6, 4), "all", (255, 0)),
])
def test_ghost_planes(n, where, counts, precision):
    rng = np.random.default_rng(sum(n) + counts[0])
    total = sum(counts)
    p = np.zeros(total, dtype=emg.PARTICLE)
    axis = rng.integers(0, 3, total)
    for d, (f, m) in enumerate(zip("xyz", n)):
        u = rng.random(total)
        last = where == "corner" or ((where == "faces") & (axis == d))
        p[f] = np.where(last, m - 1 + 0.999 * u, m * u)
    q = (0.3, -0.2)
    with emg.Context(n, q, (1.0, -1.0), (1.0, 1.0), counts, precision=precision) as ctx:
        ctx.upload(p, counts)
        rho = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3))
        ctx.charge(0, rho=rho)
    if precision == emg.PLAIN_FP64:
        ref = oracle.charge(p, counts, q, n)
        oracle.fold_rho(ref, n)
        # sums of up to 3000 terms of a node, each rounded to 2^-53
        assert np.abs(rho - ref).max() <= 1e-12 * np.abs(ref).max()
        return
    ref, size = np.zeros_like(rho), np.zeros_like(rho)
    for s in range(2):
        w = _fixed_weights(p[sum(counts[:s]):sum(counts[:s + 1])], n)
        oracle.fold_rho(w, n)
        ref += q[s] * (w / 2**24)
        size += abs(q[s]) * w / 2**24
    # whole numbers; the charges' two products and their sum round
    assert np.all(np.abs(rho - ref) <= 4 * 2.0**-53 * size)
