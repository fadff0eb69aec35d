"""The FP32 form's planning between steps (bucket capacities and starts, spill
counts, by one look-back scan) at its edges: fewer buckets than a block, one
more than a block, many blocks, with spilled particles, across a re-bucketing,
and replayed from a HIP graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_first():
    """torch has to see the device before the library initialises it."""
    import torch
    torch.cuda.is_available()


def _setup(n, ppc, vth, seed=3):
    from ctca_amd import emg
    rng = np.random.default_rng(seed)
    cnt = int(ppc * n[0] * n[1] * n[2])
    rec = np.zeros(2 * cnt, dtype=emg.PARTICLE)
    for c, name in enumerate("xyz"):
        rec[name] = rng.random(2 * cnt) * n[c]
    for name in ("vx", "vy", "vz"):
        rec[name] = rng.normal(size=2 * cnt) * vth
    rec["pid"] = np.arange(2 * cnt)
    return rec, [cnt, cnt]


# 2 species; tiles of 4 or 8 cells: 54, 256, 128, 2 x 129 = 258, 2,880, 16,384, 1,024 (twice), 1,296 and 1,024 buckets
@pytest.mark.parametrize("n,tile,ppc,vth", [
    ((12, 12, 12), 4, 6.0, 0.3),
    ((16, 16, 32), 4, 6.0, 0.05),
    ((16, 16, 16), 4, 40.0, 0.1),      # few tiles of several 1024-thread rounds
    ((12, 172, 4), 4, 6.0, 0.3),
    ((40, 96, 24), 4, 4.0, 0.45),      # fast: about 3% of the particles spill
    ((256, 256, 64), 8, 0.5, 0.3),     # sparse 8^3 tiles (256-thread blocks)
    ((64, 64, 64), 8, 8.9, 0.05),      # just under the sparse rule's 4,608 per bucket
    ((64, 64, 64), 8, 9.1, 0.05),      # just over it
    ((66, 65, 57), 8, 4.0, 0.45),      # sparse, partial tiles, staged outboxes overflow
    ((32, 32, 32), 0, 4.0, 0.45),       # the default tile of a small grid
])
def test_steps_keep_every_particle_where_it_should_be(n, tile, ppc, vth):
    from ctca_amd import emg
    rec, counts = _setup(n, ppc, vth)
    with emg.Context(n, [1.0, -1.0], [0.0, 0.0], [1.0, 1.0], counts, precision=emg.FP32_FIXED,
                     tile=tile, track_pid=True) as ctx:
        ctx.upload(rec, counts)
        ctx.set_fields(np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6)))
        x = np.stack([rec[c] for c in "xyz"], 1)
        v = np.stack([rec["v" + c] for c in "xyz"], 1)
        steps = 0
        for k in (3, 1, 2):
            for _ in range(k):
                ctx.push_es(2)
            steps += k
            rho = ctx.rho()
            rhos = [ctx.rho(species=s) for s in range(2)]
            ctx.sort()                         # a re-bucketing between steps
            ctx.deposit_rho(0)
            # integer weights: independent of the buckets the particles lie in
            assert np.array_equal(ctx.rho(), rho)
            for s in range(2):                 # free streaming: no particle lost
                assert abs(rhos[s]).sum() == pytest.approx(counts[s], rel=1e-12)
        got, cnt = ctx.download()
    assert list(cnt) == counts
    assert np.array_equal(np.sort(got["pid"]), rec["pid"])
    back = np.empty_like(got)
    back[got["pid"]] = got
    box = np.array(n, dtype=np.float64)
    want = x + 2.0 * steps * v.astype(np.float32)
    d = np.stack([back[c] for c in "xyz"], 1) - want
    d -= box * np.round(d / box)
    # an FP32 offset in [0, 1) is rounded once per step (2^-24 at most, and
    # 2^-23 of a move of a few cells), and once on upload
    assert np.abs(d).max() <= (steps + 1) * 2.0 ** -23 * max(4.0, 12.0 * vth)


def test_plan_replayed_from_a_graph():
    """Eight captured steps (the first after a re-bucketing, so nine plans),
    replayed three times with eager steps between, against eager steps."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("the library initialised the device before torch")
    from ctca_amd import emg
    n = (40, 48, 48)
    rec, counts = _setup(n, 3.0, 0.5)
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))

    def make():
        ctx = emg.Context(n, [1.0, -1.0], [0.0, 0.0], [1.0, 1.0], counts,
                          precision=emg.FP32_FIXED, tile=4)
        r = rec.copy()
        r["pid"] = 0
        ctx.upload(r, counts)
        ctx.set_fields(eb)
        ctx.synchronize()
        return ctx

    ref = make()
    want = []
    for _ in range(3):
        for _ in range(8):
            ref.push_es(2)
        want.append(ref.rho())
        for _ in range(2):
            ref.push_es(2)
        want.append(ref.rho())
    ref.close()
    ctx = make()
    st = torch.cuda.Stream()
    emg.lib().emg_set_stream(ctx.h, st.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        graph.capture_begin()
        for _ in range(8):
            ctx.push_es(2)
        graph.capture_end()
    got = []
    for _ in range(3):
        with torch.cuda.stream(st):
            graph.replay()
        got.append(ctx.rho())
        for _ in range(2):
            ctx.push_es(2)
        got.append(ctx.rho())
    ctx.synchronize()
    ctx.close()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,counts,tile", [
    ((16, 16, 16), (1, 0), 4),
    ((16, 12, 8), (2049, 2047), 4),          # chunk edges
    ((40, 40, 40), (30000, 4097), 4),        # many tiles, few particles in each
    ((128, 128, 64), (5000, 20000), 4),      # as many tiles as LDS counters, and more
    ((128, 104, 80), (5000, 20000), 4),
    ((24, 24, 24), (8388609, 10), 8),        # past the flat scatter's particles
])
def test_upload_reaches_the_buckets(n, counts, tile):
    """Every uploaded particle in its bucket: the charge of each species and the
    records that come back."""
    from ctca_amd import emg
    rng = np.random.default_rng(sum(counts))
    total = sum(counts)
    rec = np.zeros(total, dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.integers(0, m * 4096, total) / 4096.0   # exact in FP32
    rec["vx"] = np.arange(total) % 4093 / 4096.0
    rec["pid"] = np.arange(total)
    with emg.Context(n, [1.0, -1.0], [0.0, 0.0], [1.0, 1.0], counts, precision=emg.FP32_FIXED,
                     tile=tile, track_pid=True) as ctx:
        ctx.upload(rec, counts)
        ctx.deposit_rho(0)
        for s in range(2):
            assert abs(ctx.rho(species=s)).sum() == pytest.approx(counts[s], rel=1e-12)
        got, cnt = ctx.download()
    assert list(cnt) == list(counts)
    back = np.empty_like(got)
    back[got["pid"]] = got
    for f in ("x", "y", "z", "vx", "pid"):
        assert np.array_equal(back[f], rec[f])
