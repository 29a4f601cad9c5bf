"""Targets that a search's group view left out have no list, in either list layout: a copy of the lists over the whole
range leaves their rows alone, the adjoints take them with no neighbour and the pair loops leave their results as they
were. Searches that store table positions, and those that store particle indices after an earlier search of
table positions (many small groups, tables that do not fit, the fused search). Ranges off the list blocks of
64, and counts off the rounds of the copy (ragged n, ngmax not a multiple of its rounds). A target in two groups of
the view has the list that it has in one."""
import numpy as np
import pytest

from sphexa_amd import abi, ic
from sphexa_amd.particles import STD_FIELDS, ParticleSet

pytestmark = pytest.mark.gpu


def lattice():
    arr, spec = ic.sedov_lattice(11, seed=2)
    return arr, abi.Box.make(spec["lo"], spec["hi"], abi.PERIODIC)


def spread_supports():
    """supports from 50 to most of the particles: more tables outgrow their place, at ngmax = 300, than there is room for"""
    n, rng = 12000, np.random.default_rng(2)
    near = np.exp(rng.uniform(np.log(50), np.log(0.85 * n), n))
    x, y, z = rng.uniform(0, 1, (3, n))
    arr = dict(x=x, y=y, z=z, h=0.5 * (3 * near / (4 * np.pi * n)) ** (1 / 3), m=np.full(n, 1.0 / n), u=np.ones(n),
               vx=0 * x, vy=0 * x, vz=0 * x)
    return arr, abi.Box.make(0.0, 1.0, abi.OPEN)


class Case:
    def __init__(self, ngmax, particles=lattice):
        from sphexa_amd.lib import Workspace

        arr, self.box = particles()
        self.ws = Workspace(0)
        self.params = abi.Params.defaults(self.ws.K, ngmax=ngmax, ng0=60)
        self.ps = ParticleSet.from_host(arr, STD_FIELDS)
        self.n, self.ngmax = self.ps.n, ngmax
        self.ws.domain_sync(self.box, self.ps.sync_fields(), self.params, self.n)

    def search(self, fused=False):
        find = self.ws.find_neighbors_xmass if fused else self.ws.find_neighbors
        find(self.box, self.ps.fields(), self.params, 0, self.n, False, **({"rho": True} if fused else {}))

    def lists(self, first, last, host=False):
        import torch

        out = torch.full((last - first, self.ngmax), -1, dtype=torch.int32, device="cpu" if host else "cuda")
        self.ws.copy_neighbors(out, first, last)
        return out.cpu().numpy()

    def density_vjp(self, cot):
        import torch

        from sph_autograd import adjoint

        out = {k: torch.zeros(self.n, dtype=torch.float64, device="cuda") for k in ("x", "y", "z", "h")}
        self.ws.vjp("sphx_density_std_vjp", self.box, self.ps.fields(), self.params, 0, self.n, adjoint({"rho": cot}),
                    adjoint(out))
        return {k: v.cpu().numpy() for k, v in out.items()}

    def loops(self, chain):
        """std pair loops over the whole range, every result a sentinel before"""
        keys = ("rho", "c11", "c23", "ax", "du")
        for k in keys:
            self.ps.t[k].fill_(-7.0)
        p, f = abi.chained(self.params) if chain else self.params, self.ps.fields()
        self.ps.t["rho"].fill_(1.0)  # a density that the left-out targets keep
        self.ws.pair("sphx_density_std", self.box, f, p, 0, self.n)
        self.ws.eos("sphx_eos_std", f, self.params, 0, self.n)
        self.ws.pair("sphx_iad_std", self.box, f, p, 0, self.n)
        return {k: self.ps.host(k).copy() for k in ("rho", "c11", "c23")}

    def view(self, width, every):
        """groups of `width` consecutive particles, one in `every`; the mask of their targets"""
        import torch

        self.start = torch.arange(0, self.n, width * every, dtype=torch.int32, device="cuda")
        self.end = torch.clamp(self.start + width, max=self.n)
        chosen = np.zeros(self.n, bool)
        for a, b in zip(self.start.cpu().numpy(), self.end.cpu().numpy()):
            chosen[a:b] = True
        return chosen

    def set_view(self):
        view = abi.Groups(firstBody=0, lastBody=self.n, numGroups=self.start.numel())
        view.groupStart, view.groupEnd = self.start.data_ptr(), self.end.data_ptr()
        self.ws.set_groups(view)


@pytest.mark.parametrize("layout,ngmax", [(kind, n) for kind in ("tables", "many_groups", "fused") for n in (90, 150)] +
                         [("overflow", 300)])
def test_left_out_targets_have_no_list(layout, ngmax):
    import torch

    # (many groups: of 4, every second: 8 per block of 64, more than whose tables are kept)
    c = Case(ngmax, spread_supports if layout == "overflow" else lattice)
    c.search()
    whole, stored = c.lists(0, c.n), np.minimum(c.ps.host("nc").astype(np.int64) - 1, ngmax)
    assert np.array_equal((whole >= 0).sum(1), stored) and np.all(whole[:, 0] >= 0)
    np.testing.assert_array_equal(c.lists(70, c.n - 3), whole[70:c.n - 3])
    every = c.loops(chain=False)

    chosen = c.view(4 if layout == "many_groups" else 64, 2)
    rng = np.random.default_rng(1)
    cot = torch.from_numpy(np.where(chosen, rng.standard_normal(c.n), 0.0)).cuda()
    want = c.density_vjp(cot)

    c.set_view()
    c.search(fused=layout == "fused")
    c.ws.set_groups(None)
    for host in (False, True):
        some = c.lists(0, c.n, host)
        np.testing.assert_array_equal(some[chosen], whole[chosen])
        assert np.all(some[~chosen] == -1)
    got = c.density_vjp(cot)
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    plain, chained = c.loops(chain=False), c.loops(chain=True)
    np.testing.assert_array_equal(plain["rho"][chosen], every["rho"][chosen])
    assert np.all(plain["rho"][~chosen] == 1.0)
    for k in ("c11", "c23"):
        assert np.all(plain[k][~chosen] == -7.0) and not np.any(plain[k][chosen] == -7.0)
    for k in plain:
        np.testing.assert_array_equal(chained[k], plain[k], err_msg=k)


@pytest.mark.parametrize("width,step", [(64, 40), (30, 15)])  # 34 and 89 groups: tables, and particle indices below
@pytest.mark.parametrize("tiny", [False, True])
def test_targets_in_two_groups(width, step, tiny):
    """a view whose groups overlap: every target is searched, and its list is that of one group"""
    import torch

    c = Case(150)
    if tiny:
        width, step = 8, 5
    c.search()
    whole, nc, rho = c.lists(0, c.n), c.ps.host("nc").copy(), c.loops(chain=False)["rho"]
    c.start = torch.arange(0, c.n, step, dtype=torch.int32, device="cuda")
    c.end = torch.clamp(c.start + width, max=c.n)
    c.set_view()
    c.search()
    c.ws.set_groups(None)
    np.testing.assert_array_equal(c.ps.host("nc"), nc)
    np.testing.assert_array_equal(c.lists(0, c.n), whole)
    np.testing.assert_array_equal(c.loops(chain=False)["rho"], rho)
