"""The search's matrix tests against the oracle's lists, entry by entry: pairs at the very edge of the support (where
the tile is tested again exactly), far offsets and scales of the coordinates, smoothing lengths that differ
widely within a group, and a dense cluster."""
import numpy as np
import pytest

from sphexa_amd import abi
from sphexa_amd.particles import STD_FIELDS, ParticleSet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["lattice_edge", "spread_h", "far", "tiny", "huge", "coincident", "cluster"])
def test_lists_equal_the_oracles(case):
    import torch

    from oracle import oracle as O
    from oracle import pipeline
    from sphexa_amd.lib import Workspace

    ws = Workspace(0)
    rng = np.random.default_rng(4)
    side = 24
    g = (np.arange(side) + 0.5) / side
    x, y, z = (c.ravel() for c in np.meshgrid(g, g, g, indexing="ij"))
    n = x.size
    h = np.full(n, 1.25 / side)
    lo, hi = 0.0, 1.0
    if case == "lattice_edge":
        h = np.full(n, 1.0 / side)  # 2h exactly two lattice spacings: whole shells of pairs on the edge
    else:
        x, y, z = (c + rng.uniform(-0.3, 0.3, n) / side for c in (x, y, z))
    if case == "spread_h":
        h = h * rng.choice([0.3, 0.6, 1.0, 1.2], n)
    if case == "cluster":
        # nine tenths in a small ball: groups around it reach hundreds of leaves, found by the batch and one at a time
        ball = rng.permutation(n) < n * 9 // 10
        x, y, z = (np.where(ball, 0.5 + 0.02 * rng.standard_normal(n), rng.uniform(0, 1, n)) for _ in range(3))
        r2 = (x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2
        density = 0.9 * n * np.exp(-r2 / (2 * 0.02**2)) / (2 * np.pi * 0.02**2) ** 1.5 + 0.1 * n
        h = 0.5 * (300 / (4 * np.pi * density)) ** (1 / 3)
    if case == "far":
        x, y, z, lo, hi = x + 1e6, y + 1e6, z + 1e6, 1e6 - 0.1, 1e6 + 1.1
    if case in ("tiny", "huge"):
        f = 1e-18 if case == "tiny" else 1e22
        x, y, z, h, lo, hi = x * f, y * f, z * f, h * f, -0.1 * f, 1.1 * f
    if case == "coincident":
        x[1::2], y[1::2], z[1::2] = x[::2], y[::2], z[::2]
    arr = dict(x=x, y=y, z=z, h=h, m=np.full(n, 1.0 / n), u=np.ones(n), vx=0 * x, vy=0 * x, vz=0 * x)
    box = abi.Box.make(lo, hi, abi.PERIODIC if case in ("lattice_edge", "spread_h") else abi.OPEN)
    params = abi.Params.defaults(ws.K)
    o = pipeline.run(O.load("orc"), arr, box, params, form="search", iterate_h=False)
    ps = ParticleSet.from_host(arr, STD_FIELDS)
    ws.domain_sync(box, ps.sync_fields(), params, n)
    ws.find_neighbors(box, ps.fields(), params, 0, n, False)
    lists = torch.zeros(n, params.ngmax, dtype=torch.int32, device="cuda")
    ws.copy_neighbors(lists, 0, n)
    np.testing.assert_array_equal(ps.host("nc"), o["a"]["nc"])
    stored = np.minimum(ps.host("nc").astype(np.int64) - 1, params.ngmax)
    got, ref = lists.cpu().numpy().view(np.uint32), np.asarray(o["nbrs"]).reshape(n, params.ngmax)
    used = np.arange(params.ngmax)[None, :] < stored[:, None]
    assert used.any()
    np.testing.assert_array_equal(got[used], ref[used])


@pytest.mark.parametrize("boundary", [abi.PERIODIC, abi.OPEN])
@pytest.mark.parametrize("value", [np.nan, -np.nan, np.inf])
@pytest.mark.parametrize("what", ["x", "z", "h"])
def test_particle_that_is_not_finite(what, value, boundary):
    """a particle with a coordinate or smoothing length that is not a number is nobody's neighbour, and has none; the
    others' lists are those of the same search without it. An infinite coordinate is likewise out of every reach."""
    import torch

    from sphexa_amd.lib import Workspace

    if what == "h" and np.isinf(value):
        pytest.skip("an infinite support holds every particle")
    side = 20
    rng = np.random.default_rng(9)
    g = (np.arange(side) + 0.5) / side
    x, y, z = (c.ravel() + rng.uniform(-0.3, 0.3, side**3) / side for c in np.meshgrid(g, g, g, indexing="ij"))
    n = x.size
    arr = dict(x=x, y=y, z=z, h=np.full(n, 1.25 / side), m=np.full(n, 1.0 / n), u=np.ones(n), vx=0 * x, vy=0 * x, vz=0 * x)
    box = abi.Box.make(0.0, 1.0, boundary)
    ws = Workspace(0)
    params = abi.Params.defaults(ws.K)
    ps = ParticleSet.from_host(arr, STD_FIELDS)
    ws.domain_sync(box, ps.sync_fields(), params, n)

    def lists():
        out = torch.full((n, params.ngmax), -1, dtype=torch.int32, device="cuda")
        ws.find_neighbors(box, ps.fields(), params, 0, n, False)
        ws.copy_neighbors(out, 0, n)
        return out.cpu().numpy(), ps.host("nc").astype(np.int64) - 1

    # the particles go bad after the sync, as in a run that diverges between two syncs: each in another group
    bad = np.array([5, 700, 3001, n - 1])
    before, count = lists()
    ps.t[what][torch.from_numpy(bad).cuda()] = value
    after, countAfter = lists()
    np.testing.assert_array_equal(countAfter[bad], 0)
    is_bad = np.isin(np.arange(n), bad)
    for i in np.flatnonzero(~is_bad):
        want = before[i, : count[i]]
        if what != "h":
            want = want[~np.isin(want, bad)]
        np.testing.assert_array_equal(after[i, : countAfter[i]], want, err_msg=str(i))
