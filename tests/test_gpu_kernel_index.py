"""The pair loops' kernel function over the sinc indices its variants serve: 6 (unrolled polynomial), other
integers and a non-integer (FP64: the tables; FP32: generic powers), against the oracle's tables of that index.

Bars: FP64 fields 1e-10 of their largest magnitude (the kernel value is held to 2e-15 of W(0)); mixed
density 1e-5, accelerations 1e-4, as for the default index."""
import numpy as np
import pytest

from sphexa_amd import abi, ic
from sphexa_amd.particles import VE_FIELDS, ParticleSet, ideal_gas_cv, ve_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("index", [2.0, 3.0, 5.0, 6.0, 6.5, 9.0])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("side", [5, 16])  # 125 particles: supports wider than half the box; 4096: common
def test_ve_pass_at_sinc_index(monkeypatch, index, mixed, side):
    from oracle import oracle as O
    from oracle import pipeline
    from sphexa_amd.lib import Workspace

    orc = O.load("orc")
    tables = O.tables
    monkeypatch.setattr(O, "tables", lambda lib, n=6.0, dtype=np.float64: tables(lib, index, dtype))
    arr, spec = ic.turbulence_box(side, seed=4)
    arr["temp"] = arr.pop("u") / ideal_gas_cv(10.0, 5.0 / 3.0)
    box = abi.Box.make(spec["lo"], spec["hi"], abi.PERIODIC)
    ws = Workspace(0, sinc_index=index)
    params = abi.Params.defaults(ws.K, hydro_type=abi.SPHX_F32 if mixed else abi.SPHX_F64, minDt=1e-4)
    o = pipeline.run(orc, arr, box, abi.Params.defaults(ws.K, minDt=1e-4), form="ve")
    ps = ParticleSet.from_host(arr, VE_FIELDS, mixed=mixed)
    ve_step(ws, ps, box, params)
    for k in ("xm", "kx", "gradh", "c11", "divv", "ax", "ay", "az", "du"):
        ref = o["a"][k]
        err = np.max(np.abs(ps.host(k) - ref)) / np.max(np.abs(ref))
        bar = 1e-10 if not mixed else 1e-5 if k in ("xm", "kx") else 1e-4 if k in ("ax", "ay", "az") else 1e-3
        assert err <= bar, (k, err)
