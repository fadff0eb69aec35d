"""The transforms of a field solve on a grid that goes to hipFFT run on the
context's stream, also after it has changed."""
import fake_hip
import numpy as np
import pytest


def test_fft_plans_follow_the_context_stream(tmp_path):
    fake_hip.run(tmp_path, """
        n = (112, 112, 8)
        with emg.Context(n, [1.0], [1.0], [1.0], (10,)) as c:
            c.upload(records(10, n), (10,))
            c.deposit_rho(0)
            first = launches(c.solve_es, 0.0)
            assert "hipfftExecD2Z" in first and "hipfftExecZ2D" in first
            assert len([k for k in first if k.startswith("hipfftSetStream")]) == 2
            for stream in (0x1230, 0x4560):
                got = launches(emg.lib().emg_set_stream, c.h, stream)
                assert got == [f"hipfftSetStream {stream:#x}"] * 2
            own = launches(emg.lib().emg_set_stream, c.h, None)
            assert len(own) == 2 and own[0] == own[1] and own[0] != got[0]
    """)


@pytest.mark.gpu
def test_library_solve_after_the_stream_has_changed():
    """On the context's own stream, on another one, and on a new one of its own."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("the library initialised the device before torch")
    import oracle
    from ctca_amd import emg
    n, count = (112, 112, 8), 50000
    rng = np.random.default_rng(17)
    rec = np.zeros(count, dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        rec[c] = rng.random(count) * m
    stream = torch.cuda.Stream()
    phi = []
    with emg.Context(n, [0.01], [1.0], [1.0], (count,), precision=emg.FP32_FIXED) as ctx:
        ctx.upload(rec, (count,))
        for k in range(3):
            if k > 0:
                emg.lib().emg_set_stream(ctx.h, stream.cuda_stream if k == 1 else None)
            ctx.deposit_rho(0)
            ctx.solve_es(-0.01)
            phi.append(ctx.potential())
        rho = ctx.rho()
    assert np.array_equal(phi[0], phi[1]) and np.array_equal(phi[0], phi[2])
    want = oracle.fields.poisson_periodic(rho - 0.01)
    # the transforms round to some 1e-15 of the largest value
    assert np.abs(phi[0] - want).max() <= 1e-12 * np.abs(want).max()
