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


def test_a_field_solve_relocates_b_where_a_replay_may_meet_another_one(tmp_path):
    fake_hip.run(tmp_path, """
        n, counts = (16, 16, 16), (2000, 1000)
        for precision in (emg.PLAIN_FP64, emg.FP32_FIXED):
            with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts,
                             precision=precision) as c:
                def all_nodes(f, *a):
                    return "k_relocate" in launches(f, *a)

                c.upload(records(3000, n), counts)
                c.set_fields(np.zeros((19, 19, 19, 6)))
                c.push_es(2)
                assert not all_nodes(c.solve_es, 0.0)  # B is that of set_fields
                fake.fake_capture(1)
                assert all_nodes(c.solve_es, 0.0)
                fake.fake_capture(0)
                assert not all_nodes(c.solve_es, 0.0)
                c.bfield()
                fake.fake_capture(1)
                c.grdcrt()                             # recorded, not done
                fake.fake_capture(0)
                assert all_nodes(c.solve_es, 0.0)
                assert not all_nodes(c.solve_es, 0.0)
                fake.fake_capture(1)
                c.bfield()
                fake.fake_capture(0)
                c.grdcrt()
                assert all_nodes(c.solve_es, 0.0)      # a replay may have been here
    """)


def test_an_adjoint_step_allocates_nothing_after_the_window_has_begun(tmp_path):
    fake_hip.run(tmp_path, """
        n, counts = (16, 16, 16), (200000, 1000)
        for begin in (lambda c: c.adj_reset(), lambda c: c.adj_field()):
            with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts) as c:
                c.upload(records(201000, n), counts)
                c.set_fields(np.zeros((19, 19, 19, 6)))
                begin(c)
                before = fake.fake_mallocs()
                fake.fake_capture(1)
                c.adj_step(2)
                fake.fake_capture(0)
                assert fake.fake_mallocs() == before
    """)


def test_charge_and_faces_are_computed_anew_where_a_replay_may_have_moved_particles(tmp_path):
    fake_hip.run(tmp_path, """
        n, counts = (16, 16, 16), (2000, 1000)
        ghosts = ((-1,) * 3, (17,) * 3)
        for precision in (emg.PLAIN_FP64, emg.FP32_FIXED):
            for moves_alone in (False, True):
                with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts,
                                 precision=precision) as c:
                    def faces():
                        return any("faces" in k for k in launches(c.rho, *ghosts))

                    c.upload(records(3000, n), counts)
                    c.set_fields(np.zeros((19, 19, 19, 6)))
                    c.push_es(2)
                    assert launches(c.deposit_rho, 0) == []
                    assert faces() and not faces()
                    fake.fake_capture(1)
                    c.positn(2) if moves_alone else c.push_es(2)
                    deposit = launches(c.deposit_rho, 0)
                    fake.fake_capture(0)
                    assert (deposit != []) == moves_alone
                    assert (launches(c.deposit_rho, 0) != []) == moves_alone
                    assert faces() and faces()
    """)
