"""Which calls report what the particle kernels have flagged on the device: the
ones on particles and their sums, not a read-out of the potential."""
import fake_hip


def test_the_potential_leaves_the_particles_errors_to_other_calls(tmp_path):
    fake_hip.run(tmp_path, """
        n = (40, 30, 20)
        with emg.Context(n, [1.0], [1.0], [1.0], (1000,)) as c:
            c.upload(records(1000, n), (1000,))
            c.set_fields(np.zeros((23, 33, 43, 6)))
            c.deposit_rho(0)
            c.solve_es(0.0)
            for call in (c.synchronize, c.rho, c.fields, c.download):
                fake.fake_flags(4, 0)      # a particle has moved too far
                c.potential()
                with pytest.raises(emg.EmgError) as e:
                    call()
                assert e.value.code == -5
                call()
    """)
