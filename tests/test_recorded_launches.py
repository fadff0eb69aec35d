"""A program may record steps into a HIP graph, then upload, sort or update
fields, and replay: what a call launches must not depend on what the calls
before it left behind on the host."""
import fake_hip


def test_fp32_steps_launch_the_same_after_every_change_of_the_particles(tmp_path):
    fake_hip.run(tmp_path, """
        n, counts = (16, 16, 16), (2000, 1000)
        for em in (False, True):
            with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts,
                             precision=emg.FP32_FIXED) as c:
                c.upload(records(3000, n), counts)
                c.set_fields(np.zeros((19, 19, 19, 6)))
                push = c.push_em if em else c.push_es
                first = launches(push, 2)
                assert launches(push, 2) == first
                new = [dict(count=k, vth_perp=0.1, vth_para=0.1) for k in counts]
                for change in (lambda: c.upload(records(3000, n), counts), c.sort, c.download,
                               lambda: c.init_device(new, 1)):
                    change()
                    assert launches(push, 2) == first
    """)
