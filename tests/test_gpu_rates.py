"""Relaxation rates other than the reference's: the collision reads all 19 populations, so
these lattices keep the population kernels at every size.  The x march with the density
summed inside the collide (lattices the 8 x 32 tiles and the chunks cover) and with the
separate density pass, chunks of 2 to 32 planes, against the FP64 oracle; then the
one-thread-per-node collide of small FP64-storage lattices."""
import numpy as np
import pytest

import gpu_cases as gc
import oracle_lib as orc

pytestmark = pytest.mark.gpu

# a rate of their own on rows that the reference relaxes at 1 (heat-flux-like and third-order
# rows); rows 3, 5, 7 are conserved and take no rate
TS = orc.reference_ts(0.8)
for row, rate in ((1, 1.05), (10, 1.2), (12, 0.9), (16, 1.1), (18, 0.95)):
    TS[row] = rate

GEOMS = {
    # covered by the tiles: two in y and z, periodic; one z tile, walls 2 + 4
    "64x16x64": dict(dims=(64, 16, 64), eos="RKE", tr=0.60, nwall=0, spheres=[(20, 8, 31.5, 10), (43, 8, 33, 10)]),
    "32x24x32": dict(dims=(32, 24, 32), eos="PRM", tr=0.70, nwall=2, nwall_hi=4, spheres=[(16, 12, 2, 9)]),
    # partial tiles and a short last chunk
    "33x13x40": dict(dims=(33, 13, 40), eos="PRW", tr=0.70, nwall=3, spheres=[(16, 6, 3, 8)]),
}
STEPS = 60


def pair(cpmp, name, form):
    spec = GEOMS[name]
    nx, ny, nz = spec["dims"]
    kw = dict(eos=spec["eos"], tr=spec["tr"], nwall=spec["nwall"], nwall_hi=spec.get("nwall_hi"), ts=TS)
    o = orc.Oracle(orc.make_params(nx, ny, nz, **kw))
    g = cpmp.Lattice(cpmp.make_params(nx, ny, nz, form=form, **kw))
    dg, dl = gc.densities(spec["eos"], spec["tr"])
    rho = gc.sphere_rho(nx, ny, nz, spec["spheres"], 5.0, dg, dl).reshape(nx, ny, nz)
    rho[:, :, :spec["nwall"]] = 0
    rho[:, :, nz - spec.get("nwall_hi", spec["nwall"]):nz] = 0
    for s in (o, g):
        s.set_wall_mu(-0.01, 0.01)
        s.init_from_rho(rho.ravel())
    return o, g


@pytest.mark.parametrize("xc", [2, 4, 16, 32, "v1"])
@pytest.mark.parametrize("form,tol", [("fp64", 1e-10), ("fp32", 2e-4), ("fp32a", 2e-4), ("fp16", 2e-2)])
@pytest.mark.parametrize("name", list(GEOMS))
def test_other_rates_match_oracle(cpmp, monkeypatch, name, form, tol, xc):
    """the tolerances of the reference-rate runs (test_gpu_production.py) at fewer steps"""
    monkeypatch.setenv("CPMP_COLLIDE", "v1" if xc == "v1" else "march")
    if xc != "v1":
        monkeypatch.setenv("CPMP_XC", str(xc))
    print(f"[rates] {name} {form} {xc}", flush=True)
    o, g = pair(cpmp, name, form)
    fluid = o.get(orc.TYPE) == 1
    o.step(STEPS)
    # split, so that both the step within a run and the last of a call run
    for n in (1, 2, STEPS - 3):
        g.step(n)
    ro, r = o.get(orc.RHO)[fluid], g.get("rho")[fluid]
    err = gc.rel_err(r, ro) if form == "fp64" else np.max(np.abs(r - ro)) / np.max(ro)
    f = g.get("f").reshape(19, -1)[:, fluid]
    summed = np.max(np.abs(f.sum(axis=0) - r)) / np.max(r)
    print(f"[rates] {name} {form} {xc}: rho err {err:.2e}, rho - sum f {summed:.2e}", flush=True)
    assert err < tol
    assert summed < (1e-13 if form == "fp64" else 2e-6)
    if form == "fp64":
        fo = o.get(orc.F).reshape(19, -1)[:, fluid]
        assert np.max(np.abs(f - fo)) < tol * np.max(np.abs(fo))
    g.close()


def test_the_rates_are_taken(cpmp):
    """the rates of their own change the run by more than the tolerances above, in the
    oracle and on the device alike"""
    o, g = pair(cpmp, "32x24x32", "fp64")
    spec = GEOMS["32x24x32"]
    ref = orc.Oracle(orc.make_params(*spec["dims"], eos=spec["eos"], tr=spec["tr"], nwall=2, nwall_hi=4))
    ref.set_wall_mu(-0.01, 0.01)
    ref.init_from_rho(g.get("rho"))
    for s in (o, g, ref):
        s.step(STEPS)
    fluid = o.get(orc.TYPE) == 1
    ro, rr = o.get(orc.RHO)[fluid], ref.get(orc.RHO)[fluid]
    assert np.max(np.abs(ro - rr)) / np.max(ro) > 1e-4
    assert gc.rel_err(g.get("rho")[fluid], ro) < 1e-10
    g.close()
