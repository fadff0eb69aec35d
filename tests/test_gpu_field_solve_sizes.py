"""The periodic field solve over grid sizes: planes that fit in LDS and lines of
every kind of radix, and the sizes next to those limits."""
import numpy as np
import pytest

import oracle
from ctca_amd import emg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_first():
    """torch has to see the device before the library initialises it."""
    import torch
    torch.cuda.is_available()


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


@pytest.mark.parametrize("n", [(32, 32, 32), (66, 95, 46)])   # planes, lines
def test_solve_replayed_from_a_graph(n):
    """Four captured steps with their solves (an even number: the particles'
    buffers change places every step), replayed three times with eager steps
    between, against eager steps (bitwise: the charge is fixed point)."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("the library initialised the device before torch")
    rng = np.random.default_rng(3)
    counts = (20000, 20000)
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    for f, m in zip("xyz", n):
        rec[f] = rng.random(len(rec)) * m
        rec["v" + f] = 0.05 * rng.normal(size=len(rec))

    def make():
        ctx = emg.Context(n, [1e-4, -1e-4], [-1.0, 0.01], [1.0, 1.0], counts,
                          precision=emg.FP32_FIXED)
        ctx.upload(rec, counts)
        ctx.deposit_rho(0)
        ctx.solve_es(0.0)
        ctx.synchronize()
        return ctx

    def steps(ctx, k):
        for _ in range(k):
            ctx.push_es(2)
            ctx.solve_es(0.0)

    ref, want = make(), []
    for _ in range(3):
        for k in (4, 2):
            steps(ref, k)
            want.append(ref.potential())
    ref.close()
    ctx, got = make(), []
    st = torch.cuda.Stream()
    emg.lib().emg_set_stream(ctx.h, st.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        graph.capture_begin()
        steps(ctx, 4)
        graph.capture_end()
    for _ in range(3):
        with torch.cuda.stream(st):
            graph.replay()
        got.append(ctx.potential())
        steps(ctx, 2)
        got.append(ctx.potential())
    ctx.synchronize()
    ctx.close()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
