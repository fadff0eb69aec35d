"""The adjoint kernels with a particle that a push has left outside the box (and
reported): every access stays in the grid."""
import numpy as np
import pytest

from ctca_amd import emg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("sign", [-1.0, 1.0])
def test_adjoint_step_after_a_reported_far_move(axis, sign):
    n, count = (8, 12, 10), 500
    rng = np.random.default_rng(axis)
    rec = np.zeros(count, dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(count) * m
    rec["v" + "xyz"[axis]][::100] = sign * 2.5 * n[axis]
    g = rng.normal(size=n[::-1])
    with emg.Context(n, [1.0], [0.5], [1.0], (count,)) as ctx:
        ctx.upload(rec, (count,))
        ctx.set_fields(np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6)))
        ctx.positn(1)
        with pytest.raises(emg.EmgError) as e:
            ctx.synchronize()
        assert e.value.code == -5
        ctx.adj_reset()
        ctx.adj_add_density(g, (1.0,))
        ctx.adj_step(2)
        assert np.isfinite(ctx.adj_velocity_sums()).all()
        assert np.isfinite(ctx.adj_field()).all()
