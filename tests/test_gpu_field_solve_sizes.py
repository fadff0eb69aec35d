"""The periodic field solve over grid sizes: planes that fit in LDS and lines of
every kind of radix, and the sizes next to those limits."""
import numpy as np
import pytest

import oracle
from ctca_amd import emg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [
    (2, 2, 2), (3, 2, 5), (2, 3, 64), (4, 16, 8), (16, 4, 9),
    (32, 32, 32), (64, 64, 64), (15, 13, 11), (17, 19, 61), (53, 7, 3), (24, 40, 6),
    (77, 63, 14), (90, 70, 9), (7, 26, 22),
    (67, 8, 8), (8, 8, 211), (8, 223, 8),  # the largest radix, and a prime above it
    (100, 97, 8),              # the largest plane that LDS holds, and one above
    (100, 98, 8),
    (111, 97, 10), (95, 66, 8), (19, 510, 4), (512, 38, 6),   # x lines in ragged groups
    (12, 10, 512), (6, 10, 640),
])
@pytest.mark.parametrize("precision", [emg.PLAIN_FP64, emg.FP32_FIXED])
def test_solve_matches_numpy(n, precision):
    if precision == emg.FP32_FIXED and min(n) < 4:
        pytest.skip("the FP32 form needs four cells per axis")
    rng = np.random.default_rng(sum(n))
    counts = (4000, 3000)
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    for f, m in zip("xyz", n):
        rec[f] = rng.random(len(rec)) * m
    bk = 0.003
    back = 0.01 * rng.normal(size=n[::-1])
    with emg.Context(n, [0.01, -0.02], [1.0, -1.0], [1.0, 1.0], counts,
                     precision=precision) as ctx:
        ctx.upload(rec, counts)
        for step in range(2):
            if step:
                ctx.set_background(back)
            ctx.deposit_rho(0)
            rho = ctx.rho() + bk + step * back
            ctx.solve_es(bk)
            phi = ctx.potential()
            ref = oracle.fields.poisson_periodic(rho)
            # the transforms' passes, of at most 211 terms, round to some
            # 1e-15 of the largest value
            assert np.abs(phi - ref).max() <= 1e-12 * np.abs(ref).max()
