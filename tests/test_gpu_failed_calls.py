"""What a workspace holds after a call that failed: nothing of an earlier one stands in for it."""
import numpy as np
import pytest

from sphexa_amd import abi, ic
from sphexa_amd.particles import STD_FIELDS, ParticleSet

pytestmark = pytest.mark.gpu


@pytest.fixture()
def case():
    from sphexa_amd.lib import Workspace

    arr, spec = ic.sedov_lattice(16, seed=4)
    ws = Workspace(0)
    box = abi.Box.make(spec["lo"], spec["hi"], abi.PERIODIC)
    ps = ParticleSet.from_host(arr, STD_FIELDS)
    params = abi.Params.defaults(ws.K)
    ws.domain_sync(box, ps.sync_fields(), params, ps.n)
    ws.find_neighbors(box, ps.fields(), params, 0, ps.n, False)
    ws.pair("sphx_density_std", box, ps.fields(), params, 0, ps.n)
    return ws, box, ps, params


def code_of(call):
    from sphexa_amd.lib import SphxError

    with pytest.raises(SphxError) as e:
        call()
    return e.value.code


def test_keys_out_of_order(case):
    """no tree is left by a build that refused its keys: a search says so, until the next build"""
    import torch

    ws, box, ps, params = case
    nc = ps.host("nc").copy()
    keys = ps.t["keys"][: ps.n].clone()
    assert code_of(lambda: ws.build_tree(torch.flip(keys, (0,)).contiguous(), box)) == abi.SPHX_ERR_ARG
    search = lambda: ws.find_neighbors(box, ps.fields(), params, 0, ps.n, False)  # noqa: E731
    assert code_of(search) == abi.SPHX_ERR_STATE
    assert code_of(ws.tree_view) == abi.SPHX_ERR_STATE
    ws.build_tree(keys, box)
    search()
    np.testing.assert_array_equal(ps.host("nc"), nc)


@pytest.mark.parametrize("fused", [False, True])
def test_search_without_room_for_its_lists(case, fused):
    """lists of 2^30 entries a target (TiB) cannot be allocated: the search reports it and the pair loops and copies say
    that there are no lists, rather than reading the former ones' memory; a later search works"""
    ws, box, ps, params = case
    nc, rho = ps.host("nc").copy(), ps.host("rho").copy()
    large = abi.Params.from_buffer_copy(params)
    large.ngmax = 1 << 30
    find, out = (ws.find_neighbors_xmass, dict(rho=True)) if fused else (ws.find_neighbors, {})
    assert code_of(lambda: find(box, ps.fields(), large, 0, ps.n, False, **out)) == abi.SPHX_ERR_ALLOC
    out = ps.t["nc"].new_zeros(ps.n * params.ngmax)
    assert code_of(lambda: ws.copy_neighbors(out, 0, ps.n)) == abi.SPHX_ERR_STATE
    assert code_of(lambda: ws.pair("sphx_density_std", box, ps.fields(), params, 0, ps.n)) == abi.SPHX_ERR_STATE
    ws.find_neighbors(box, ps.fields(), params, 0, ps.n, False)
    ws.pair("sphx_density_std", box, ps.fields(), params, 0, ps.n)
    np.testing.assert_array_equal(ps.host("nc"), nc)
    np.testing.assert_array_equal(ps.host("rho"), rho)


def test_refused_search_keeps_the_lists(case):
    """a search refused for its arguments has touched nothing: the former lists serve on"""
    ws, box, ps, params = case
    rho = ps.host("rho").copy()
    wrong = abi.Params.from_buffer_copy(params)
    wrong.ng0 = wrong.ngmax + 1
    assert code_of(lambda: ws.find_neighbors(box, ps.fields(), wrong, 0, ps.n, False)) == abi.SPHX_ERR_ARG
    # (the std fields hold no xm)
    assert code_of(lambda: ws.find_neighbors_xmass(box, ps.fields(), params, 0, ps.n, False)) == abi.SPHX_ERR_ARG
    ws.pair("sphx_density_std", box, ps.fields(), params, 0, ps.n)
    np.testing.assert_array_equal(ps.host("rho"), rho)
