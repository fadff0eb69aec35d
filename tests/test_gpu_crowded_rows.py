"""emg_sort on grids with more blocks of a run length than cells: that run table
stays unbuilt and its kernels keep their plain slices.  (The re-sorts of
sort_every order patches, whose tables are always built.)"""
import fake_hip
import numpy as np
import pytest

CASES = [(20000, 2), (150000, 1), (400000, 0)]   # particles on 4^3 cells, tables built


@pytest.mark.parametrize("count,tables", CASES)
def test_tables_built_by_a_sort_of_rows(tmp_path, count, tables):
    fake_hip.run(tmp_path, f"""
        n, counts = (4, 4, 4), ({count}, {count} // 5)
        with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts) as c:
            c.upload(records(sum(counts), n), counts)
            assert launches(c.sort).count("k_run_fill") == {tables}
    """)


@pytest.mark.gpu
@pytest.mark.parametrize("count,tables", CASES)
def test_pushes_after_a_sort_of_rows_equal_unsorted_ones(count, tables):
    from ctca_amd import emg
    n, counts = (4, 4, 4), (count, count // 5)
    rng = np.random.default_rng(count)
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(len(rec)) * m
        rec["v" + c] = rng.normal(size=len(rec)) * 0.05
    rec["pid"] = np.arange(len(rec))
    core = rng.normal(size=(n[2], n[1], n[0], 6)) * 0.01
    at = [np.arange(-1, v + 2) % v for v in n]
    eb = np.ascontiguousarray(core[np.ix_(at[2], at[1], at[0])])
    out = []
    for rows in (False, True):
        with emg.Context(n, [0.002, -0.002], [1.0, -0.01], [1.0, 1.0], counts) as ctx:
            ctx.upload(rec, counts)
            ctx.set_fields(eb)
            got = []
            for em in (False, True):
                if rows:
                    ctx.sort()
                for _ in range(2):
                    ctx.push_em(2) if em else ctx.push_es(2)
                got.append(ctx.current() if em else ctx.rho())
            ctx.deposit_rho(0)
            got.append(ctx.rho())
            p, _ = ctx.download()
        out.append((got, p[np.argsort(p["pid"], kind="stable")]))
    for f in ("x", "y", "z", "vx", "vy", "vz", "pid"):
        assert np.array_equal(out[0][1][f], out[1][1][f]), f
    # sums of up to 8 count / 64 terms in another order, each rounded at 2^-49 or
    # 2^-53 of the largest
    for a, b in zip(out[0][0], out[1][0]):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()
