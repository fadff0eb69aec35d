"""Grids that get 4^3 tiles because 8^3 ones would be fewer than the chip's CUs:
what 8^3 tiles keep, they keep (twice as many particles leave a tile of 4, or
pass the cell beyond it)."""
import numpy as np
import pytest

from ctca_amd import emg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count,sigma,drift", [
    ((16, 16, 16), 400 * 4096, 0.2, 0.0),    # dense: most movers overflow the outboxes
    ((32, 32, 32), 4 * 32768, 0.0, 1.7),     # a beam: one in six passes the cell beyond
    ((18, 13, 27), 250 * 6318, 0.12, 0.0),   # partial tiles
])
@pytest.mark.parametrize("em", [False, True])
def test_movers_that_fit_with_tiles_of_8_fit_with_the_default(n, count, sigma, drift, em):
    rng = np.random.default_rng(count)
    rec = np.zeros(count, dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(count) * m
        rec["v" + c] = rng.normal(size=count) * (sigma / 2)
    rec["vx"] += drift / 2
    got = []
    for tile in (0, 8):
        with emg.Context(n, [1.0], [0.0], [1.0], (count,), precision=emg.FP32_FIXED,
                         tile=tile) as ctx:
            ctx.upload(rec, (count,))
            ctx.set_fields(np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6)))
            for _ in range(3):
                ctx.push_em(2) if em else ctx.push_es(2)
                ctx.synchronize()
            got.append(ctx.current() if em else ctx.rho())
    assert np.array_equal(*got)              # integer sums
    if not em:
        assert got[0].sum() == pytest.approx(count, rel=1e-9)
