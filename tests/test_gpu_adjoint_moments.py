"""The FP64 adjoint on the step on moments: the tape written by it, checkpoints restored into
it, runs of it on the second stream.  Lattices of 80 000 nodes and more take it by
themselves; the schedule tests of test_gpu_adjoint.py run on it by CPMP_COLLIDE=moments."""
import numpy as np
import pytest

import oracle_lib as orc
import test_gpu_adjoint as ta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,hi,scheme", [(3, 3, 1), (4, 3, 0)])
def test_adjoint_of_a_lattice_on_moments_matches_the_oracle(cpmp, monkeypatch, lo, hi, scheme):
    """92 160 nodes: J and the gradients against the oracle's reverse mode, all steps taped,
    recomputed from checkpoints, and both with a call before it on the same context"""
    monkeypatch.delenv("CPMP_COLLIDE", raising=False)
    dims, nsteps = (48, 48, 40), 8
    kw, rho0, mu_lo, mu_hi, target = ta.small_case(cpmp, *dims)
    kw.update(nwall=lo, nwall_hi=hi, wall_scheme=scheme)
    o = orc.Oracle(orc.make_params(*dims, **kw))
    o.set_wall_mu(mu_lo, mu_hi)
    o.init_from_rho(rho0)
    Jo, glo_o, ghi_o, gka_o = o.adjoint(nsteps, target)
    g = cpmp.Lattice(cpmp.make_params(*dims, **kw))
    assert g.memory() > (2 * 19 + 12) * 8 * rho0.size     # holds a moment set
    g.set_wall_mu(mu_lo, mu_hi)
    for every, budget in ((3, 0), (8, -1), (2, 3 * 80 * rho0.size)):
        g.init_from_rho(rho0)
        J, glo, ghi, gka = g.adjoint(nsteps, target, checkpoint_every=every, tape_budget_bytes=budget)
        assert J == pytest.approx(Jo, rel=1e-10)
        assert np.max(np.abs(glo - glo_o)) < 1e-7 * np.max(np.abs(glo_o))
        assert np.max(np.abs(ghi - ghi_o)) < 1e-7 * np.max(np.abs(ghi_o)) + 1e-12
        assert gka == pytest.approx(gka_o, rel=1e-7)
        assert np.allclose(g.get("rho"), o.get(orc.RHO), rtol=1e-10)
    # the state is left where the run went, and goes on from there as an undisturbed one
    h = cpmp.Lattice(cpmp.make_params(*dims, **kw))
    h.set_wall_mu(mu_lo, mu_hi)
    h.init_from_rho(rho0)
    h.step(nsteps)
    for lat in (g, h):
        lat.step(3)
    assert np.array_equal(g.get("rho"), h.get("rho")) and np.array_equal(g.get("f"), h.get("f"))
    g.close()
    h.close()


@pytest.mark.parametrize("dims", [(16, 12, 20), (18, 14, 33)])
@pytest.mark.parametrize("schedule", ["budget", "interval", "limit", "overlap", "repeat"])
def test_schedules_agree_on_moments(cpmp, monkeypatch, schedule, dims):
    monkeypatch.setenv("CPMP_COLLIDE", "moments")
    if schedule == "limit":
        return ta.test_adjoint_memory_limit_sub_segments_agree(cpmp)
    if schedule == "overlap":
        return ta.test_adjoint_overlapped_schedule_matches_serial(cpmp, monkeypatch, "fp64", dims)
    per_step = 80 * dims[0] * dims[1] * dims[2]
    calls = {"budget": [(6, 0), (6, 13 * per_step), (6, -1)], "interval": [(1, 0), (5, 0), (40, 0)],
             "repeat": [(6, 0), (40, -1), (1, 0), (7, 9 * per_step), (6, 0)]}[schedule]
    g, target = ta._small_lattice(cpmp, dims)
    rho0, res = g.get("rho"), []
    for every, budget in calls:
        if schedule != "repeat":
            g.close()
            g, target = ta._small_lattice(cpmp, dims)
        g.init_from_rho(rho0)
        g.step(2)       # moments are current when the call begins
        res.append(g.adjoint(40, target, checkpoint_every=every, tape_budget_bytes=budget) + (g.get("rho"),))
    g.close()
    for r in res[1:]:
        assert r[0] == res[0][0] and r[3] == res[0][3]
        for i in (1, 2, 4):
            assert np.array_equal(r[i], res[0][i])


def test_moments_and_populations_give_the_same_gradients(cpmp, monkeypatch):
    """the forward run on moments against the one-thread-per-node kernels: 40 steps apart by
    rounding, and so are the gradients of the two trajectories"""
    res = {}
    for collide in ("moments", "v1"):
        monkeypatch.setenv("CPMP_COLLIDE", collide)
        g, target = ta._small_lattice(cpmp, (16, 12, 20))
        res[collide] = g.adjoint(40, target, checkpoint_every=7)
        g.close()
    a, b = res["moments"], res["v1"]
    assert a[0] == pytest.approx(b[0], rel=1e-10) and a[3] == pytest.approx(b[3], rel=1e-7)
    for i in (1, 2):
        assert np.max(np.abs(a[i] - b[i])) < 1e-7 * np.max(np.abs(b[i]))
