"""The adjoint step's transposed gather, binned by tiles: against a plain FP64
torch restatement, on grids with partial tiles, fewer cells than a tile, one
tile per axis, more tiles than a workgroup counts in LDS, and with populations
of both slice lengths and of several passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_first():
    """torch has to see the device before the library initialises it."""
    import torch
    torch.cuda.is_available()


def _corners(x, n):
    import torch
    i = torch.minimum(x.long(), torch.tensor([v - 1 for v in n], device=x.device))
    f = x - i
    for q in range(8):
        o = [(q >> d) & 1 for d in range(3)]
        g = [(i[:, d] + o[d]) % n[d] for d in range(3)]
        s = [1.0 if o[d] else -1.0 for d in range(3)]
        w = [f[:, d] if o[d] else 1.0 - f[:, d] for d in range(3)]
        grad = torch.stack([s[0] * w[1] * w[2], w[0] * s[1] * w[2], w[0] * w[1] * s[2]], 1)
        yield (g[2] * n[1] + g[1]) * n[0] + g[0], w[0] * w[1] * w[2], grad


def _reference(parts, node, g, n, qm, qfac):
    """One adj_add_density(g), one adj_step(2), one adj_add_density(g), one
    adj_step(2): the two nodal fields and the velocity sums."""
    import torch
    ncell = n[0] * n[1] * n[2]
    fields, sums = [], []
    lam = []
    for x, q in zip(parts, qfac):
        lx = sum(g[idx][:, None] * gr for idx, _, gr in _corners(x, n)) * q
        lam.append([lx, torch.zeros_like(lx)])
    for step in range(2):
        acc = torch.zeros((ncell, 3), dtype=torch.float64, device=g.device)
        for s, x in enumerate(parts):
            lx, lv = lam[s]
            qmp = qm[s]  # qm ustep / 2
            bf = sum(w[:, None] * node[idx][:, 3:] for idx, w, _ in _corners(x, n))
            w3 = lv + 2.0 * lx
            b = -qmp * bf
            bor = 2.0 / (1.0 + (b * b).sum(1, keepdim=True))
            mt = w3 + bor * torch.linalg.cross(w3 + torch.linalg.cross(w3, b), b)
            la = mt + w3
            for idx, w, gr in _corners(x, n):
                lx = lx + qmp * (la * node[idx][:, :3]).sum(1)[:, None] * gr
                acc.index_add_(0, idx, (qmp * w)[:, None] * la)
            if step == 0:
                lx = lx + sum(g[idx][:, None] * gr for idx, _, gr in _corners(x, n)) * qfac[s]
            lam[s] = [lx, mt]
        fields.append(acc)
    return fields, torch.stack([l[1].sum(0) for l in lam])


@pytest.mark.parametrize("n,counts", [
    ((8, 8, 8), (300, 5)),                       # one tile, its own neighbour
    ((5, 20, 3), (4000, 1)),                     # fewer cells than a tile
    ((17, 9, 33), (30000, 0)),                   # partial tiles, an empty species
    ((136, 136, 128), (60000, 20000)),           # 4,624 tiles: no LDS counters
    ((24, 30, 16), (2 ** 21 + 77, 4096)),        # long slices
    ((16, 16, 16), (2 ** 24 - 100, 2 ** 20)),    # two passes
])
def test_adjoint_step_against_fp64_torch(n, counts):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("the library initialised the device before torch")
    from ctca_amd import emg
    rng = np.random.default_rng(sum(n) + counts[0])
    q, qm = [0.01, -0.02], [1.0, -0.3]
    box = np.array(n, dtype=np.float64)
    rec = np.zeros(sum(counts), dtype=emg.PARTICLE)
    pos = rng.random((len(rec), 3)) * box
    pos[: min(3, len(pos))] = [[0.0, 0.0, 0.0], box - 1e-9, box][: min(3, len(pos))]
    for c, name in enumerate("xyz"):
        rec[name] = pos[:, c]
    eb = np.zeros((n[2] + 3, n[1] + 3, n[0] + 3, 6))
    core = rng.normal(size=(n[2], n[1], n[0], 6)) * 0.05
    at = [(np.arange(-1, v + 2) % v) for v in n]
    eb[...] = core[np.ix_(at[2], at[1], at[0])]
    gsc = rng.normal(size=(n[2], n[1], n[0]))
    with emg.Context(n, q, qm, [1.0, 1.0], counts, precision=emg.PLAIN_FP64) as ctx:
        ctx.upload(rec, counts)
        ctx.set_fields(eb)
        ctx.adj_reset()
        ctx.adj_add_density(gsc, q)
        ctx.adj_step(2)
        f0 = ctx.adj_field()
        ctx.adj_add_density(gsc, q)
        ctx.adj_step(2)
        f1 = ctx.adj_field()
        sums = ctx.adj_velocity_sums()
    dev = "cuda"
    c = torch.from_numpy(core).to(dev)

    def back(a, d):
        return torch.roll(a, 1, 2 - d)

    node = [0.5 * (c[..., d] + back(c[..., d], d)) for d in range(3)]
    for d in range(3):
        u, w = [a for a in range(3) if a != d]
        b = c[..., 3 + d]
        node.append(0.25 * (b + back(b, u) + back(b, w) + back(back(b, u), w)))
    node = torch.stack(node, -1).reshape(-1, 6)
    x = torch.from_numpy(pos).to(dev)
    parts = [x[: counts[0]], x[counts[0]:]]
    fields, want = _reference(parts, node, torch.from_numpy(gsc).to(dev).reshape(-1), n, qm, q)
    # both sides are FP64 sums of the same terms in another order: a node's
    # sum of k terms is within k eps of the sum of their sizes
    k = 8 * max(64.0, sum(counts) / (n[0] * n[1] * n[2]))
    for got, ref in zip((f0, f1), fields):
        ref = ref.reshape(n[2], n[1], n[0], 3).cpu().numpy()
        assert np.abs(got - ref).max() <= 4 * k * 2.2e-16 * np.abs(ref).max() + 1e-300
    ref = want.cpu().numpy()
    assert np.abs(sums - ref).max() <= 1e-10 * max(1.0, np.abs(ref).max())
