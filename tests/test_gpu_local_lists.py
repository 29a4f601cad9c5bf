"""Neighbour lists as table positions and the pair loops' record sources: staged tables, tables of other groups
than the call's, tables that do not fit, and the FP32 form's fixed point in boxes of several shapes.

Lists and counts are compared entry by entry; results of one search over different target ranges and
groupings bit for bit; fields against the oracle at the repository's bars (FP64 1e-10 of the field's
largest magnitude; mixed density 1e-5, accelerations 1e-4)."""
import numpy as np
import pytest

from sphexa_amd import abi, ic
from sphexa_amd.particles import GRADV_FIELDS, STD_FIELDS, VE_FIELDS, ParticleSet, ideal_gas_cv, std_step, ve_step

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ws():
    from sphexa_amd.lib import Workspace

    return Workspace(0)


def std_loops(ws, ps, box, params, ranges):
    f = ps.fields()
    for a, b in ranges:
        ws.pair("sphx_density_std", box, f, params, a, b)
    ws.eos("sphx_eos_std", f, params, 0, ps.n)
    for a, b in ranges:
        ws.pair("sphx_iad_std", box, f, params, a, b)
    for a, b in ranges:
        ws.momentum_energy_std(box, f, params, a, b)
    return {k: ps.host(k).copy() for k in ("rho", "c11", "c23", "ax", "ay", "az", "du")}


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [63, 64, 65, 129, 4096, 5000])
def test_ranges_of_one_search_bitwise(ws, mixed, n):
    """blocks whose targets' lists lie in two tables (ranges off the search's groups) give the same bits"""
    arr, box = ic.evrard_sphere(n, seed=n)
    arr["vx"] = 0.1 * np.sin(6.0 * arr["x"])
    box = abi.Box.make(box["lo"], box["hi"], abi.OPEN)
    params = abi.Params.defaults(ws.K, hydro_type=abi.SPHX_F32 if mixed else abi.SPHX_F64)
    ps = ParticleSet.from_host(arr, STD_FIELDS, mixed=mixed)
    std_step(ws, ps, box, params)
    whole = std_loops(ws, ps, box, params, [(0, n)])
    cut = std_loops(ws, ps, box, params, [(0, n // 3), (n // 3, n - 7), (n - 7, n)])
    for k, v in whole.items():
        np.testing.assert_array_equal(cut[k], v, err_msg=k)


def kernel_sum(arr, h, lists, count, periodic, K):
    """m_i + sum_j m_j W(r_ij / h_i) times K / h_i^3 over the lists, W = sinc^6(pi v / 2), in 64 bits"""
    x, m = np.stack([arr[k] for k in "xyz"], 1), arr["m"]
    rho = np.empty(len(h))
    for i in range(len(h)):
        j = lists[i, : count[i]]
        d = x[j] - x[i]
        d -= np.round(d) if periodic else 0.0
        v = np.minimum(np.sqrt((d * d).sum(1)) / h[i], 2.0)
        rho[i] = K / h[i] ** 3 * (m[i] + (m[j] * np.sinc(v / 2.0) ** 6).sum())
    return rho


def check_search(arr, box, mixed, iterate, searches=1, **params):
    """h, counts and the kept entries of a search equal the oracle's, and so does the density over them"""
    import torch

    from oracle import oracle as O
    from oracle import pipeline
    from sphexa_amd.lib import Workspace

    ws = Workspace(0)  # (what a search needed, the next ones on its workspace start with)
    hydro = np.float32 if mixed else np.float64
    arr = dict(arr, h=arr["h"].astype(hydro), m=arr["m"].astype(hydro))
    ps = ParticleSet.from_host(arr, STD_FIELDS, mixed=mixed)
    params = abi.Params.defaults(ws.K, hydro_type=ps.hydro_type, **params)
    o = pipeline.run(O.load("orc"), arr, box, params, form="search", iterate_h=iterate, hydro=hydro)
    ws.domain_sync(box, ps.sync_fields(), params, ps.n)
    f, h = ps.fields(), ps.t["h"].clone()
    for _ in range(searches):
        ps.t["h"].copy_(h)
        assert ws.find_neighbors(box, f, params, 0, ps.n, iterate) == (o["fails"] == 0)
        # the device's pow in the update of h may differ by an ulp from the C library's; a float's can move pairs over
        # the edge of the support
        np.testing.assert_allclose(ps.host("h"), o["a"]["h"], rtol=4 * np.finfo(hydro).eps if iterate else 0, atol=0)
        same = not (iterate and mixed)
        np.testing.assert_allclose(ps.host("nc").astype(np.int64), o["a"]["nc"].astype(np.int64), atol=0 if same else 1, rtol=0)
        lists = torch.zeros(ps.n, params.ngmax, dtype=torch.int32, device="cuda")
        ws.copy_neighbors(lists, 0, ps.n)
        got, ref = lists.cpu().numpy(), np.asarray(o["nbrs"]).reshape(ps.n, -1).view(np.int32)
        count = np.minimum(ps.host("nc").astype(np.int64) - 1, params.ngmax)
        if same:
            used = np.arange(params.ngmax)[None, :] < count[:, None]
            np.testing.assert_array_equal(got[used], ref[used])
        ws.pair("sphx_density_std", box, f, params, 0, ps.n)
        rho = kernel_sum({k: ps.host(k) for k in ("x", "y", "z", "m")}, ps.host("h").astype(np.float64), got, count,
                         box.boundary[0] == abi.PERIODIC, ws.K)
        # FP64: the 20000-point table's interpolant, 6e-9 of W(0) a term; mixed: FP32 separations
        np.testing.assert_allclose(ps.host("rho"), rho, rtol=1e-5 if mixed else 2e-7)
    return ps


@pytest.mark.parametrize("mixed", [False, True])
def test_lists_full_long_before_the_support(mixed):
    """supports of 4000 neighbours, far over ngmax: the first ngmax in visiting order are kept, the rest counted"""
    arr, spec = ic.turbulence_box(20, seed=3)
    arr["h"] = arr["h"] * 3.5
    box = abi.Box.make(spec["lo"], spec["hi"], abi.PERIODIC)
    ps = check_search(arr, box, mixed, False)
    assert ps.host("nc").min() > 2049


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,ngmax", [(6000, 300), (12000, 235), (12000, 300), (12000, 400)])
def test_tables_that_outgrow_their_place(n, ngmax, mixed):
    """supports from 50 to most of the particles: groups with more than the 2048 or 2496 particles that a table has room for,
    by turns few enough for the regions that the first search finds, for those that its repetition is given, and too
    many (the lists then hold particle indices). Each search twice, as by a later step"""
    rng = np.random.default_rng(2)
    near = np.exp(rng.uniform(np.log(50), np.log(0.85 * n), n))
    x, y, z = rng.uniform(0, 1, (3, n))
    arr = dict(x=x, y=y, z=z, h=0.5 * (3 * near / (4 * np.pi * n)) ** (1 / 3), m=rng.uniform(0.5, 1.5, n) / n,
               u=np.ones(n), vx=0 * x, vy=0 * x, vz=0 * x)
    check_search(arr, abi.Box.make(0.0, 1.0, abi.OPEN), mixed, False, 2, ngmax=ngmax)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("some", [1, 16])
def test_tables_of_an_iteration(some, mixed):
    """smoothing lengths off by up to a factor of 3, for all targets or one in 16: the h iteration searches a group's
    targets several times, each round adding to the table that the lists of the finished ones refer to"""
    rng = np.random.default_rng(7)
    n = 9000
    x, y, z = rng.uniform(0, 1, (3, n))
    h = 0.5 * (3 * 200 / (4 * np.pi * n)) ** (1 / 3) * np.where(rng.integers(0, some, n) == 0, 3.0 ** rng.uniform(-1, 1, n), 1.0)
    arr = dict(x=x, y=y, z=z, h=h, m=np.full(n, 1.0 / n), u=np.ones(n), vx=0 * x, vy=0 * x, vz=0 * x)
    check_search(arr, abi.Box.make(0.0, 1.0, abi.PERIODIC), mixed, True, 2, ng0=200, ngmax=300)


@pytest.mark.parametrize("lengths,boundary", [((1.0, 1.0, 0.5), abi.PERIODIC),
                                              ((1.0, 1.0, 0.5), [abi.PERIODIC, abi.PERIODIC, abi.OPEN]),
                                              ((1.0, 0.7, 0.5), abi.OPEN)])
def test_mixed_box_shapes(ws, lengths, boundary):
    """the fixed point with one unit for all dimensions (one periodic length, or none) and without (several)"""
    from oracle import oracle as O
    from oracle import pipeline

    side = [int(24 * v) for v in lengths]
    rng = np.random.default_rng(8)
    g = np.meshgrid(*[(np.arange(s) + 0.5) / 24.0 for s in side], indexing="ij")
    x, y, z = (c.ravel() + rng.uniform(-0.1, 0.1, c.size) / 24.0 for c in g)
    n = x.size
    arr = dict(x=x, y=y, z=z, h=np.full(n, 1.44 / 24.0), m=np.full(n, 1.0 / n), vx=0.1 * np.sin(6 * x),
               vy=0.1 * np.cos(5 * y), vz=0.05 * z, alpha=np.full(n, 0.3),
               temp=np.full(n, 1.0 / ideal_gas_cv(10.0, 5.0 / 3.0)))
    box = abi.Box.make([0.0] * 3, list(lengths), boundary)
    o = pipeline.run(O.load("orc"), arr, box, abi.Params.defaults(ws.K, minDt=1e-4), form="ve")
    ps = ParticleSet.from_host(arr, VE_FIELDS, mixed=True)
    ve_step(ws, ps, box, abi.Params.defaults(ws.K, hydro_type=abi.SPHX_F32, minDt=1e-4))
    np.testing.assert_array_equal(ps.host("nc"), o["a"]["nc"])
    for k, bar in (("xm", 1e-5), ("kx", 1e-5), ("ax", 1e-4), ("ay", 1e-4), ("az", 1e-4), ("du", 1e-4)):
        ref = o["a"][k]
        err = np.max(np.abs(ps.host(k) - ref)) / np.max(np.abs(ref))
        assert err <= bar, (k, err)


@pytest.mark.parametrize("index", [6.0, 5.0])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("side", [4, 5, 10, 17])  # 64, 125, 1000 and 4913 targets: supports wider than half the box first
def test_gathered_records_bitwise(index, mixed, side):
    """the VE loops over particle indices (left by the fused search), whose records come from global memory, give the bits
    of those over table positions, whose records are staged; with the AV cleaning, and without"""
    from sphexa_amd.lib import Workspace

    arr, spec = ic.turbulence_box(side, seed=6)
    arr["temp"] = arr.pop("u") / ideal_gas_cv(10.0, 5.0 / 3.0)
    box = abi.Box.make(spec["lo"], spec["hi"], abi.PERIODIC)
    ws = Workspace(0, sinc_index=index)
    ps = ParticleSet.from_host(arr, VE_FIELDS + GRADV_FIELDS, mixed=mixed)
    params = abi.Params.defaults(ws.K, hydro_type=ps.hydro_type, minDt=1e-4)
    n, f = ps.n, ps.fields()
    alpha = ps.t["alpha"].clone()
    ws.domain_sync(box, ps.sync_fields(), params, n)
    result = {}
    for fused in (False, True):
        (ws.find_neighbors_xmass if fused else ws.find_neighbors)(box, f, params, 0, n, False)
        ps.t["alpha"].copy_(alpha)
        for loop in ("sphx_xmass", "sphx_ve_def_gradh"):
            ws.pair(loop, box, f, params, 0, n)
        ws.eos("sphx_eos_ve", f, params, 0, n)
        for loop in ("sphx_iad_divv_curlv", "sphx_av_switches"):
            ws.pair(loop, box, f, params, 0, n)
        out = {}
        for clean in (False, True):
            ws.momentum_energy_ve(box, f, params, 0, n, clean)
            out.update({k + str(clean): ps.host(k).copy() for k in ("ax", "ay", "az", "du")})
        result[fused] = dict(out, **{k: ps.host(k).copy() for k in ("xm", "kx", "gradh", "c11", "divv", "curlv", "alpha")})
    for k, v in result[False].items():
        np.testing.assert_array_equal(result[True][k], v, err_msg=k)
