"""Uploads with records that are not alive (nid < 0): the living ones in order,
no copy of them on the host, and no error of an earlier call lost."""
import fake_hip
import pytest

DEAD, FAR = 32, 4      # device flags: a dead record met, a particle moved too far

SETUP = """
        import resource
        rng = np.random.default_rng(2)

        def sent():
            "where the records of the last transfer went: slots, pids"
            n = 4000000
            slot, pid = np.zeros(n, "i8"), np.zeros(n, "i4")
            fake.fake_split.restype = ctypes.c_int64
            k = fake.fake_split(slot.ctypes.data_as(ctypes.c_void_p),
                                pid.ctypes.data_as(ctypes.c_void_p), ctypes.c_int64(n))
            return slot[:k], pid[:k]
"""


@pytest.mark.parametrize("room", [1.0, 0.9])
@pytest.mark.parametrize("counts", [(7, 5), (3000, 1), (4096, 2048), (50000, 30000), (0, 9000)])
def test_living_records_keep_their_order(tmp_path, counts, room):
    fake_hip.run(tmp_path, SETUP + f"""
        n, counts = (12, 10, 8), np.array({counts})
        total = counts.sum()
        r = records(total, n, pid=True)
        r["nid"][rng.random(total) < 0.3] = -1
        alive = [(r["nid"][:counts[0]] >= 0).sum(), (r["nid"][counts[0]:] >= 0).sum()]
        capacity = [max(a, int(k * {room})) for a, k in zip(alive, counts)]
        with emg.Context(n, [1.0, -1.0], [1.0, 1.0], [1.0, 1.0], capacity) as c:
            fake.fake_flags({DEAD}, 0)   # of the transfer that meets them (if there is room)
            if {room} < 1.0:
                fake.fake_flags(0, 0)
            c.upload(r, counts)
            slot, pid = sent()
            assert list(c.counts()) == alive
        want = r["pid"][r["nid"] >= 0]
        # the first transfer left its other records behind the living ones
        put = dict(zip(slot, pid))
        for s in range(2):
            first = 0 if s == 0 else capacity[0]
            got = [put[first + k] for k in range(alive[s])]
            assert got == list(want[sum(alive[:s]):sum(alive[:s + 1])])
    """)


def test_no_host_copy_and_no_lost_error(tmp_path):
    fake_hip.run(tmp_path, SETUP + f"""
        n, total = (12, 10, 8), 2000000
        r = records(total, n)
        r["nid"][-1] = -1
        with emg.Context(n, [1.0], [1.0], [1.0], (total,)) as c:
            c.upload(r[:100], (100,))
            # a push has left an error on the device, reported by the upload
            fake.fake_flags({DEAD} | {FAR}, 0)
            with pytest.raises(emg.EmgError) as e:
                c.upload(r, (total,))
            assert e.value.code == -5
            assert c.counts().sum() == 0
            used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
            resource.setrlimit(resource.RLIMIT_AS, (used + (64 << 20), -1))  # records: 128 MB
            fake.fake_flags({DEAD}, 0)
            c.upload(r, (total,))
            assert c.counts().sum() == total - 1
    """)
