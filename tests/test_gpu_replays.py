"""Graphs of steps replayed after the program has changed the particles or the
fields eagerly: equal to the same calls without a graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_first():
    """torch has to see the device before the library initialises it."""
    import torch
    torch.cuda.is_available()


class Recorded:
    """What `calls` launches on a context, recorded once and replayed."""

    def __init__(self, ctx, calls):
        import torch
        from ctca_amd import emg
        self.torch, self.stream = torch, torch.cuda.Stream()
        emg.lib().emg_set_stream(ctx.h, self.stream.cuda_stream)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(self.stream):
            self.graph.capture_begin()
            calls()
            self.graph.capture_end()

    def __call__(self):
        with self.torch.cuda.stream(self.stream):
            self.graph.replay()


def need_torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("the library initialised the device before torch")


@pytest.mark.parametrize("em", [False, True])
def test_fp32_steps_recorded_after_a_step_and_replayed_after_an_upload(em):
    need_torch()
    from ctca_amd import emg
    n, counts = (24, 20, 16), (30000, 9000)
    rng = np.random.default_rng(31)
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))

    def records(part):
        """particles in `part` of the box, with moves of up to a cell or two"""
        r = np.zeros(sum(counts), dtype=emg.PARTICLE)
        for c, m in zip("xyz", n):
            r[c] = rng.random(sum(counts)) * m * part
            r["v" + c] = rng.normal(size=sum(counts)) * 0.15
        return r

    sets = [records(1.0), records(0.4), records(0.7)]

    def program(ctx, recorded):
        push = ctx.push_em if em else ctx.push_es

        def steps():
            for _ in range(4):     # an even number: two state buffers
                push(2)

        out = []
        ctx.upload(sets[0], counts)
        ctx.set_fields(eb)
        push(2)
        push(2)
        four = Recorded(ctx, steps) if recorded else steps
        for k in range(4):
            four()
            push(2)
            push(2)
            out.append(ctx.current() if em else ctx.rho())
            if k < 2:
                ctx.upload(sets[k + 1], counts)
            else:
                ctx.sort()
                ctx.sort()
        return out

    got = []
    for recorded in (False, True):
        with emg.Context(n, [1.0, -1.0], [0.0, 0.0], [1.0, 1.0], counts,
                         precision=emg.FP32_FIXED) as ctx:
            got.append(program(ctx, recorded))
    for a, b in zip(*got):         # integer sums: in any order
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_recorded_solves_replayed_after_b_updates(precision):
    need_torch()
    from ctca_amd import emg
    n, counts = (16, 20, 12), (9000, 4000)
    rng = np.random.default_rng(5)
    core = rng.normal(size=(n[2], n[1], n[0], 6)) * 0.1
    at = [np.arange(-1, v + 2) % v for v in n]
    eb = np.ascontiguousarray(core[np.ix_(at[2], at[1], at[0])])
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(sum(counts)) * m
        rec["v" + c] = rng.normal(size=sum(counts)) * 0.1

    def program(ctx, recorded):
        def steps():
            for _ in range(2):
                ctx.solve_es(0.1)
                ctx.push_es(2)

        ctx.upload(rec, counts)
        ctx.set_fields(eb)
        ctx.deposit_rho(0)
        ctx.solve_es(0.1)
        ctx.push_es(2)
        ctx.push_es(2)
        two = Recorded(ctx, steps) if recorded else steps
        two()
        ctx.set_fields(eb)     # E anew, so that B changes by its curl
        ctx.bfield()
        ctx.grdcrt()
        ctx.push_es(2)
        ctx.push_es(2)
        ctx.bfield()
        two()
        two()
        return ctx.energy(), ctx.fields()

    out = []
    for recorded in (False, True):
        with emg.Context(n, [0.02, -0.02], [1.0, -1.0], [1.0, 1.0], counts,
                         precision=emg.PLAIN_FP64 if precision == "fp64" else emg.FP32_FIXED) as c:
            out.append(program(c, recorded))
    # the same kernels: sums of atomics in another order at most (FP64), or the
    # energy's partial sums of particles in another order (FP32)
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()


def test_adjoint_steps_recorded_after_a_reset():
    need_torch()
    from ctca_amd import emg
    n, counts = (16, 20, 12), (9000, 4000)
    rng = np.random.default_rng(8)
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(sum(counts)) * m
    core = rng.normal(size=(n[2], n[1], n[0], 6)) * 0.1
    at = [np.arange(-1, v + 2) % v for v in n]
    eb = np.ascontiguousarray(core[np.ix_(at[2], at[1], at[0])])
    g = rng.normal(size=n[::-1])

    def program(ctx, recorded):
        ctx.upload(rec, counts)
        ctx.set_fields(eb)
        ctx.adj_reset()
        step = (lambda: ctx.adj_step(2))
        if recorded:
            step = Recorded(ctx, step)
        out = []
        for _ in range(3):
            ctx.adj_add_density(g, (0.5, -0.25))
            step()
            out.append(ctx.adj_velocity_sums())
            out.append(ctx.adj_field())
        return out

    got = []
    for recorded in (False, True):
        with emg.Context(n, [0.02, -0.02], [1.0, -1.0], [1.0, 1.0], counts) as ctx:
            got.append(program(ctx, recorded))
    for a, b in zip(*got):         # FP64 sums of some thousand terms in another order
        assert np.abs(a - b).max() <= 1e-11 * np.abs(a).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_ghost_planes_after_replays(precision):
    need_torch()
    from ctca_amd import emg
    n, counts = (16, 20, 12), (9000, 4000)
    rng = np.random.default_rng(6)
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(sum(counts)) * m
        rec["v" + c] = rng.normal(size=sum(counts)) * 0.2
    box = (-1,) * 3, tuple(m + 1 for m in n)

    def program(ctx, recorded):
        def steps():
            ctx.push_es(2)
            ctx.push_es(2)

        out = []
        ctx.upload(rec, counts)
        ctx.set_fields(np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6)))
        steps()
        two = Recorded(ctx, steps) if recorded else steps
        for _ in range(3):
            two()
            out.append(ctx.rho(*box))
        return out

    got = []
    for recorded in (False, True):
        with emg.Context(n, [1.0, -0.5], [0.0, 0.0], [1.0, 1.0], counts,
                         precision=emg.PLAIN_FP64 if precision == "fp64" else emg.FP32_FIXED) as c:
            got.append(program(c, recorded))
    for a, b in zip(*got):         # sums of some tens of weights in another order
        assert np.abs(a - b).max() <= 1e-13 * np.abs(a).max()
