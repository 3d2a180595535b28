"""Wall fills of every depth against the oracle: up to four layers run in one launch, as
does the simple scheme at any depth; deeper layered walls run one launch per layer."""
import numpy as np
import pytest

import gpu_cases as gc
import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("collide", ["auto", "moments"])
@pytest.mark.parametrize("scheme", [0, 1])
@pytest.mark.parametrize("lo,hi", [(1, 2), (4, 1), (2, 4), (4, 4), (5, 3), (0, 6)])
def test_wall_fill_and_its_adjoint_at_every_depth(cpmp, monkeypatch, lo, hi, scheme, collide):
    """two steps (solid density and potential included), then the adjoint of five, on a
    lattice the 16 x 16 column tiles do not cover, with the per-node collide it takes and on
    moments"""
    if collide != "auto":
        monkeypatch.setenv("CPMP_COLLIDE", collide)
    dims = (18, 17, 26)
    kw = dict(eos="VDW", tr=0.8, nwall=lo, nwall_hi=hi, wall_scheme=scheme)
    rng = np.random.default_rng(4)
    rho0 = rng.uniform(2.5, 4.0, dims).ravel()
    mw = np.linspace(-0.02, 0.02, dims[0] * dims[1])
    o = orc.Oracle(orc.make_params(*dims, **kw))
    g = cpmp.Lattice(cpmp.make_params(*dims, **kw))
    for s in (o, g):
        s.set_wall_mu(mw, 0.01)
        s.init_from_rho(rho0)
        s.step(2)
    assert gc.rel_err(g.get("rho"), o.get(orc.RHO)) < 1e-12
    assert np.max(np.abs(g.get("mu") - o.get(orc.MU))) < 1e-11 * np.max(np.abs(o.get(orc.MU)))
    target = rho0 * 1.01
    J, glo, ghi, gka = g.adjoint(5, target, checkpoint_every=2)
    Jo, glo_o, ghi_o, gka_o = o.adjoint(5, target)
    assert J == pytest.approx(Jo, rel=1e-11)
    for a, b in ((glo, glo_o), (ghi, ghi_o)):
        assert np.max(np.abs(a - b)) <= 1e-8 * max(np.max(np.abs(b)), 1e-12)
    assert gka == pytest.approx(gka_o, rel=1e-8)
    g.close()
