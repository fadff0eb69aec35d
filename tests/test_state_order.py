"""Whether a state's order keeps neighbours together, which picks the kernels of
its charge, is saved and loaded with it."""
import fake_hip


def test_saved_states_keep_their_order(tmp_path):
    fake_hip.run(tmp_path, """
        n, count = (40, 30, 20), 200000
        rec = records(count, n)

        def binned(c):
            return "k_tile_charge" in launches(c.deposit_rho, 0)

        def upload(c, ordered):
            # the device's count of near neighbours, over every eighth block
            fake.fake_flags(0, count // 8 if ordered else 0)
            c.upload(rec, (count,))

        with emg.Context(n, [1.0], [1.0], [1.0], (count,)) as c:
            upload(c, True)
            assert not binned(c)
            c.state_save(0)
            upload(c, False)
            assert binned(c)
            c.state_save(1)
            c.sort()
            c.state_save(2)
            for slot in (0, 1, 2, 1, 0):
                c.state_load(slot)
                assert binned(c) == (slot == 1), slot
    """)
