"""What a context holds on the device."""
import fake_hip


def test_uploaded_fields_are_held_once(tmp_path):
    fake_hip.run(tmp_path, """
        n = (40, 30, 20)
        for precision in (emg.PLAIN_FP64, emg.FP32_FIXED):
            with emg.Context(n, [1.0], [1.0], [1.0], (1000,), precision=precision) as c:
                before = fake.fake_used()
                fake.fake_peak(1)
                eb = np.zeros((23, 33, 43, 6))
                for _ in range(2):
                    c.set_fields(eb)
                    assert fake.fake_used() == fake.fake_peak(0) == before + eb.nbytes
    """)


def test_the_tile_records_make_room_for_other_arrays(tmp_path):
    fake_hip.run(tmp_path, """
        n, counts = (40, 30, 20), (1000000, 1000)
        rec = records(sum(counts), n)

        def context():
            c = emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], counts)
            c.upload(rec, counts)
            c.set_fields(np.zeros((23, 33, 43, 6)))
            return c

        uses = (lambda c: c.sort(), lambda c: c.state_save(0), lambda c: c.solve_es(0.0))
        for use in uses:
            with context() as c:
                if use is uses[2]:
                    c.push_es(2)                     # by the plain kernels: rho for the solve
                bare = fake.fake_used()
                use(c)
                enough = fake.fake_used()            # without the records
            with context() as c:
                c.deposit_rho(0)                     # in no order: binned by tiles
                held = fake.fake_used()
                assert held - bare >= 32 * sum(counts) or use is uses[2]
                fake.fake_limit(enough + 1000000)    # the bins' counters
                use(c)
                assert fake.fake_used() <= enough + 1000000
                fake.fake_limit(2 ** 60)
                c.upload(rec, counts)
                assert "k_tile_charge" in launches(c.deposit_rho, 0)

        # a graph that bins keeps its records
        with context() as c:
            c.deposit_rho(0)
            held = fake.fake_used()
            c.upload(rec, counts)
            fake.fake_capture(1)
            c.deposit_rho(0)
            fake.fake_capture(0)
            fake.fake_limit(held)
            with pytest.raises(emg.EmgError) as e:
                c.sort()
            assert e.value.code == -3
            fake.fake_limit(2 ** 60)
    """)
