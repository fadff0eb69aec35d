"""Device allocations that fail, one or two in a row (the second after the tile
records have made room): the call says so, or does without, and the context is as
usable afterwards as before."""
import fake_hip
import pytest

CHILD = """
    n, counts = (24, 20, 16), (200000, 1000)
    total = sum(counts)
    rec = records(total, n)
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))
    precision = {precision}
    adjoint = precision == emg.PLAIN_FP64

    def create():
        return emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts, precision=precision,
                           sort_every=2 if precision == emg.PLAIN_FP64 else 0)

    def calls(c):
        "one of each call that may allocate, as often as it takes until all has been"
        yield lambda: c.upload(rec, counts)
        yield lambda: c.deposit_rho(0)
        yield lambda: c.set_fields(eb)
        yield lambda: c.solve_es(0.0)
        yield lambda: c.field_energy(1.0)
        yield lambda: c.set_background(np.zeros(n[::-1]))
        if adjoint:
            yield lambda: c.state_save(3)
            yield lambda: c.adj_reset()
            yield lambda: c.adj_step(2)
            yield lambda: c.adj_field()
            yield lambda: c.adj_velocity_sums()
            yield lambda: c.state_load(3)
        yield lambda: c.push_es(2)
        yield lambda: c.push_em(2)
        yield lambda: c.push_es(2)
        yield c.sort
        yield c.download
        yield c.energy
        yield lambda: c.rho((-1, -1, -1))
        yield lambda: c.init_device([dict(count=k, vth_perp=0.1, vth_para=0.1) for k in counts], 1)
        yield lambda: c.push_es(2)

    with create() as c:                  # how many allocations there are
        at_create = fake.fake_mallocs()
        for f in [*calls(c), *calls(c)]:
            f()
        allocations, want = fake.fake_mallocs(), fake.fake_used()
    assert fake.fake_used() == 0

    refused = 0
    for k in range(1, allocations + 1):
        fake.fake_fail_in(k, {times})
        try:
            c = create()
        except emg.EmgError as e:
            assert e.code == -3 and k <= at_create, (k, e)
            assert fake.fake_used() == 0, k   # nothing is left of it
            continue
        for f in calls(c):
            before = c.counts()
            for _ in range({times} + 1):
                try:
                    f()
                    break                 # there is memory
                except emg.EmgError as e:
                    refused += 1
                    assert e.code == -3, (k, e)
                    assert (c.counts() == before).all(), k
            else:
                raise AssertionError(k)
        assert c.counts().sum() == total
        fake.fake_fail_in(-1, 0)
        for f in calls(c):
            f()
        # nothing is missing (the tile records are halved until they fit)
        rec = 32 * total
        assert fake.fake_used() in (want, want - rec // 2, want - rec + rec // 4 // 32 * 32), k
        c.close()
        assert fake.fake_used() == 0, k
        assert fake.fake_bad_frees() == fake.fake_bad_args() == fake.fake_bad_copies() == 0, k
    assert refused or {times} == 1
"""


@pytest.mark.parametrize("precision", ["emg.PLAIN_FP64", "emg.FP32_FIXED"])
@pytest.mark.parametrize("times", [1, 2])
def test_every_allocation_may_fail(tmp_path, precision, times):
    fake_hip.run(tmp_path, CHILD.format(precision=precision, times=times))
