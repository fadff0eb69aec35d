"""Context.charge into the caller's arrays, of whatever kind they are."""
import fake_hip


def test_charge_assigns_to_arrays_that_hand_out_copies(tmp_path):
    fake_hip.run(tmp_path, """
        class Stored:
            "an array kept elsewhere (a file): reads are copies, writes assignments"
            def __init__(self, shape):
                self.a = np.full(shape, 7.0)
                self.shape, self.dtype = self.a.shape, self.a.dtype
            def __getitem__(self, at):
                return self.a[at].copy()
            def __setitem__(self, at, v):
                self.a[at] = v

        n = (6, 5, 4)
        with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], (10, 10)) as c:
            c.upload(records(20, n), (10, 10))
            shape = (n[2] + 3, n[1] + 3, n[0] + 3)
            plain = np.full(shape, 7.0), np.full((5,) + shape, 7.0)
            masked = np.ma.masked_all(shape), np.ma.masked_all((5,) + shape)
            other = Stored(shape), Stored((5,) + shape)
            narrow = np.full(shape, 7.0, "f4"), np.full((5,) + shape, 7.0, "f4")
            for rho, rhodg in (plain, masked, other, narrow):
                c.charge(2, rho, rhodg)
                # the kernels that fill the read-outs do not run here: they hold zeros
                assert not rho[...].any() and not rhodg[...].any()
            assert not masked[0].mask.any() and not masked[1].mask.any()
    """)
