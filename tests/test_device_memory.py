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
