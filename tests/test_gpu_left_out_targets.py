"""Targets that a search's group view left out have no list: a copy of the lists over the whole range leaves their rows
alone, and the adjoints take them with no neighbour. Ranges off the list blocks of 64, and counts off the rounds of the
copy (ragged n, ngmax not a multiple of its rounds)."""
import numpy as np
import pytest

from sphexa_amd import abi, ic
from sphexa_amd.particles import STD_FIELDS, ParticleSet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ngmax", [90, 150])
def test_left_out_targets_have_no_list(ngmax):
    import torch

    from sph_autograd import adjoint
    from sphexa_amd.lib import Workspace

    arr, spec = ic.sedov_lattice(11, seed=2)
    ws = Workspace(0)
    params = abi.Params.defaults(ws.K, ngmax=ngmax, ng0=60)
    box = abi.Box.make(spec["lo"], spec["hi"], abi.PERIODIC)
    ps = ParticleSet.from_host(arr, STD_FIELDS)
    n = ps.n
    ws.domain_sync(box, ps.sync_fields(), params, n)

    def lists(first, last):
        out = torch.full((last - first, ngmax), -1, dtype=torch.int32, device="cuda")
        ws.copy_neighbors(out, first, last)
        return out.cpu().numpy()

    def density_vjp(cot):
        out = {k: torch.zeros(n, dtype=torch.float64, device="cuda") for k in ("x", "y", "z", "h")}
        ws.vjp("sphx_density_std_vjp", box, ps.fields(), params, 0, n, adjoint({"rho": cot}), adjoint(out))
        return {k: v.cpu().numpy() for k, v in out.items()}

    ws.find_neighbors(box, ps.fields(), params, 0, n, False)
    whole, stored = lists(0, n), np.minimum(ps.host("nc").astype(np.int64) - 1, ngmax)
    assert np.array_equal((whole >= 0).sum(1), stored) and np.all(whole[:, 0] >= 0)
    part = lists(70, n - 3)
    np.testing.assert_array_equal(part, whole[70:n - 3])

    start = torch.arange(0, n, 64, dtype=torch.int32, device="cuda")[::2].contiguous()
    end = torch.clamp(start + 64, max=n)
    chosen = np.zeros(n, bool)
    for a, b in zip(start.cpu().numpy(), end.cpu().numpy()):
        chosen[a:b] = True
    rng = np.random.default_rng(1)
    cot = torch.from_numpy(np.where(chosen, rng.standard_normal(n), 0.0)).cuda()
    want = density_vjp(cot)

    view = abi.Groups(firstBody=0, lastBody=n, numGroups=start.numel())
    view.groupStart, view.groupEnd = start.data_ptr(), end.data_ptr()
    ws.set_groups(view)
    ws.find_neighbors(box, ps.fields(), params, 0, n, False)
    ws.set_groups(None)
    some = lists(0, n)
    np.testing.assert_array_equal(some[chosen], whole[chosen])
    assert np.all(some[~chosen] == -1)
    got = density_vjp(cot)
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
