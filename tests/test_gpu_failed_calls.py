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
