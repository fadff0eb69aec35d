"""Host transfers through the pinned slots: sizes of one chunk, several chunks,
more chunks than slots and several threads; boxes of every kind of read-out;
uploads with dead records, more records than room, and errors that must leave
the caller's array alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _records(n, total, seed=1):
    from ctca_amd import emg
    rng = np.random.default_rng(seed)
    rec = np.zeros(total, dtype=emg.PARTICLE)
    for c, name in enumerate("xyz"):
        rec[name] = rng.random(total) * n[c]
    for name in ("vx", "vy", "vz"):
        rec[name] = rng.normal(size=total) * 0.05
    rec["pid"] = np.arange(total)
    return rec


# 64-byte records: 1, 4,096 (one chunk), 4,097 and 60,000 (a few), 131,073 and
# 400,001 (several threads, slots used again)
@pytest.mark.parametrize("counts", [(1, 0), (4095, 1), (4000, 97), (0, 60000), (131072, 1),
                                    (250001, 150000)])
@pytest.mark.parametrize("fp64", [True, False])
def test_records_up_and_down(counts, fp64):
    from ctca_amd import emg
    n = (16, 8, 24)
    rec = _records(n, sum(counts))
    with emg.Context(n, [1.0, 2.0], [1.0, -1.0], [1.0, 1.0], counts,
                     precision=emg.PLAIN_FP64 if fp64 else emg.FP32_FIXED,
                     track_pid=not fp64) as ctx:
        for _ in range(2):
            ctx.upload(rec, counts)
            got, cnt = ctx.download()
            assert list(cnt) == list(counts)
            back = np.empty_like(got)
            back[got["pid"]] = got
            assert np.array_equal(back["spec"], np.repeat([1, 2], counts))
            for name in ("x", "y", "z", "vx", "vy", "vz"):
                if fp64:
                    assert np.array_equal(got[name], rec[name])
                else:  # an offset below 1 and a velocity, rounded to FP32 once
                    assert np.abs(back[name] - rec[name]).max() <= 2.0 ** -24


@pytest.mark.parametrize("n", [(4, 4, 4), (40, 33, 30), (96, 96, 90)])
def test_boxes_of_every_read_out(n):
    """Any box equals the same part of the whole one, and ghosts are images."""
    from ctca_amd import emg
    rec = _records(n, 5000)
    rec["pid"] = 0
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))
    core = np.random.default_rng(3).normal(size=(n[2], n[1], n[0], 6)) * 1e-3
    at = [np.arange(-1, v + 2) % v for v in n]
    eb[...] = core[np.ix_(at[2], at[1], at[0])]
    lo, hi = (1, 0, 2), tuple(v - 1 for v in n)
    part = tuple(slice(lo[d], hi[d] + 1) for d in (2, 1, 0))
    with emg.Context(n, [1.0, -0.5], [1.0, -1.0], [1.0, 1.0], [3000, 2000], tile=4,
                     precision=emg.FP32_FIXED) as ctx:
        ctx.upload(rec, [3000, 2000])
        ctx.set_fields(eb)
        assert np.array_equal(ctx.fields(), eb)
        assert np.array_equal(ctx.fields(lo, hi), core[part])
        ctx.push_em(2)
        whole = ctx.current()
        assert np.array_equal(ctx.current(lo, hi), whole[part])
        ghost = ctx.current((-2, -2, -2), tuple(v + 1 for v in n))
        idx = [np.arange(-2, v + 2) % v for v in n]
        assert np.array_equal(ghost, whole[np.ix_(idx[2], idx[1], idx[0])])
        ctx.deposit_rho(2)
        whole = ctx.rho()
        assert np.array_equal(ctx.rho(lo, hi), whole[part])
        box = np.zeros(tuple(v + 3 for v in reversed(n)))
        dg = np.ones((3,) + box.shape)
        ctx.charge(2, rho=box, rhodg=dg)
        assert np.array_equal(box, ctx.rho((-1, -1, -1), tuple(v + 1 for v in n)))
        assert np.array_equal(dg[1], ctx.rho((-1, -1, -1), tuple(v + 1 for v in n), species=1))
        assert not dg[2].any()
        strided = np.zeros(box.shape + (2,))[..., 0]
        ctx.charge(0, rho=strided)
        assert np.array_equal(strided, box)
        ctx.solve_es(0.0)
        phi = ctx.potential()
        assert phi.shape == tuple(reversed(n)) and np.isfinite(phi).all()


def test_dead_records_are_dropped_and_errors_leave_the_state():
    from ctca_amd import emg
    n = (16, 16, 16)
    rec = _records(n, 150000)
    rec["nid"][10::3] = -1
    rec["x"][10] = np.nan              # a dead record is not looked at
    alive = rec[rec["nid"] >= 0]
    cnt = [100000, 50000]
    kept = [int((rec["nid"][:100000] >= 0).sum()), int((rec["nid"][100000:] >= 0).sum())]
    for cap in (cnt, kept):            # with room for all, and for the living only
        with emg.Context(n, [1.0, 1.0], [1.0, 1.0], [1.0, 1.0], cap) as ctx:
            ctx.upload(rec, cnt)
            got, c = ctx.download()
            assert list(c) == kept
            for name in ("x", "vz", "pid"):
                assert np.array_equal(got[name], alive[name])
            with pytest.raises(emg.EmgError) as e:
                ctx.upload(np.concatenate([alive, alive]),
                           [2 * kept[0], 2 * kept[1]])
            assert e.value.code == -7
            assert list(ctx.counts()) == kept      # refused before anything changed
            bad = alive.copy()
            bad["y"][70000] = 99.0
            with pytest.raises(emg.EmgError) as e:
                ctx.upload(bad, kept)
            assert e.value.code == -5
            ctx.upload(alive, kept)
            ctx.deposit_rho(0)
            assert ctx.rho().sum() == pytest.approx(sum(kept), rel=1e-12)
