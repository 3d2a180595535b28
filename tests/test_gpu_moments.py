"""Runs of steps on 13 moments per node (k_moment_step) against the population kernels.

The moments carry exactly what the collision reads at the reference's rates, so a run
must agree with the one-thread-per-node population kernels (CPMP_COLLIDE=v1) to the
rounding of its sums.  The sizes are the edges of the 12 x 32 (y, z) tiles and of the
x chunks: one row or column more or less than a tile, a tile of a single column, fewer
planes than the stencils reach, chunks of one plane and longer than the lattice, and
the one-row lattices with their own tile of 192 columns."""
import os

import numpy as np
import pytest

import gpu_cases as gc

pytestmark = pytest.mark.gpu

# dims, chunk, walls, options
CASES = [
    ((9, 12, 32), 4, 0, {}),
    ((8, 13, 33), 3, 3, {}),                    # a tile of one row, a tile of one column
    ((7, 11, 31), 7, 0, {}),                    # below one tile; nx below 8 (general wrap)
    ((1, 24, 64), 1, 0, {}),
    ((5, 25, 65), 2, 0, dict(lap_points=7)),
    ((10, 3, 40), 10, 3, dict(wall_scheme=0)),
    ((16, 14, 20), 64, 3, dict(wall_scheme=2)),
    ((12, 13, 34), 5, 3, dict(K1=0.003, K2=-0.003)),
    ((12, 23, 24), 5, 3, dict(forcing=1)),
    ((12, 13, 34), 5, 0, dict(forcing=1, K1=0.003, K2=-0.003)),
    ((13, 2, 40), 5, 3, {}),                    # rows that are each other's neighbours on both sides
    ((7, 4, 33), 3, 0, {}),
    ((20, 1, 191), 6, 3, {}),
    ((6, 1, 193), 1, 0, {}),
    ((11, 1, 385), 4, 3, dict(forcing=1)),
]


def lattice(cpmp, monkeypatch, case, form, collide):
    dims, xc, nwall, opts = case
    monkeypatch.setenv("CPMP_COLLIDE", collide)
    monkeypatch.setenv("CPMP_XC", str(xc))
    g = cpmp.Lattice(cpmp.make_params(*dims, eos="VDW", tr=0.8, nwall=nwall, form=form, **opts))
    monkeypatch.delenv("CPMP_COLLIDE")
    monkeypatch.delenv("CPMP_XC")
    if nwall:
        g.set_wall_mu(0.002, 0.01)
    rng = np.random.default_rng(7)
    nx, ny, nz = dims
    rho = 3.5 + 0.3 * rng.standard_normal(dims)
    rho[:, :, :nwall] = rho[:, :, nz - nwall:] = 0
    g.init_from_rho(rho.ravel())
    return g


@pytest.mark.parametrize("form,tol", [("fp64", 1e-12), ("fp32", 1e-5), ("fp32a", 1e-5)])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])))
def test_moment_runs_match_the_population_kernels(cpmp, monkeypatch, case, form, tol):
    """7 steps from rough densities (every node differs from its neighbours, so a value
    taken from a wrong node shows at once).  A step sums 19 values and the moments once
    more, some 40 roundings of at most the largest population: 7 * 40 * 2^-53 = 3e-14
    (FP64) and 1.7e-5 / 2 (FP32) relative to the density, and smaller in practice."""
    a = lattice(cpmp, monkeypatch, case, form, "moments")
    b = lattice(cpmp, monkeypatch, case, form, "v1")
    a.step(7)
    b.step(7)
    fluid = a.get("type") == 1
    for field in ("rho", "f", "mv", "mu"):
        x, y = a.get(field).reshape(-1, fluid.size)[:, fluid], b.get(field).reshape(-1, fluid.size)[:, fluid]
        scale = np.max(np.abs(b.get("rho"))) if field in ("rho", "f") else max(np.max(np.abs(y)), 0.1)
        err = np.max(np.abs(x - y)) / scale
        print(f"[moments] {case[0]} {form} {field}: {err:.2e}", flush=True)
        assert err < tol, field
    a.close()
    b.close()


@pytest.mark.parametrize("form", ["fp64", "fp32", "fp32a"])
@pytest.mark.parametrize("case", [CASES[1], CASES[7], CASES[8], CASES[10], CASES[12]], ids=lambda c: "x".join(map(str, c[0])))
def test_moment_runs_split_into_calls_are_bitwise_the_same(cpmp, monkeypatch, tmp_path, case, form):
    """the populations between calls lose nothing: one call of 6 steps, and calls of
    1 + 2 + 3 steps with a checkpoint taken into another lattice in between"""
    a = lattice(cpmp, monkeypatch, case, form, "moments")
    b = lattice(cpmp, monkeypatch, case, form, "moments")
    c = lattice(cpmp, monkeypatch, case, form, "moments")
    a.step(6)
    b.step(1)
    b.step(2)
    path = str(tmp_path / "split.ckp")
    b.checkpoint_save(path)
    c.checkpoint_load(path)
    c.step(3)
    for field in ("rho", "mu", "f", "mv"):
        assert np.array_equal(a.get(field), c.get(field)), field
    for g in (a, b, c):
        g.close()


@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[10], CASES[12]], ids=lambda c: "x".join(map(str, c[0])))
def test_fp32_arithmetic_form_sums_the_density_in_fp64(cpmp, monkeypatch, case):
    """FP64 storage with FP32 arithmetic: the stored density is the FP64 sum of the 19
    values that the next step pulls, from the sums of two (one rounding of 2^-24 each) and
    of four (two) that the moments use anyway.  Sums of all 19 in FP32 err by 0.3 to 0.5
    of 2^-24 of the density on average, these by 0.1."""
    a = lattice(cpmp, monkeypatch, case, "fp32a", "moments")
    fluid = a.get("type") == 1
    u = 2.0 ** -24
    for n in (1, 4):
        a.step(n)
        f = a.get("f").reshape(19, -1)[:, fluid]
        err = np.abs(a.get("rho")[fluid] - f.sum(axis=0))
        bound = u * (np.abs(f[1:7]).sum(axis=0) + 2 * np.abs(f[7:]).sum(axis=0)) + 36 * 2.0 ** -53 * np.abs(f).sum(axis=0)
        mean = float(np.mean(err / f.sum(axis=0))) / u
        print(f"[moments] {case[0]} fp32a density: {np.max(err / bound):.2f} of the bound, mean {mean:.2f} 2^-24", flush=True)
        assert np.all(err <= bound)
        assert mean < 0.2
    a.close()


@pytest.mark.parametrize("form", ["fp64", "fp32", "fp32a"])
def test_the_switches_select_the_path(cpmp, monkeypatch, form):
    """CPMP_COLLIDE=moments takes the moments on a lattice of any size, =march the population
    march, and CPMP_XC changes the chunk only: told apart by the moment set, 12 values per
    node and more, in the lattice's memory"""
    dims, n, word = (64, 16, 64), 64 * 16 * 64, 8 if form == "fp64" else 4

    def memory(collide, xc):
        for k, v in (("CPMP_COLLIDE", collide), ("CPMP_XC", xc)):
            monkeypatch.setenv(k, v) if v else monkeypatch.delenv(k, raising=False)
        g = cpmp.Lattice(cpmp.make_params(*dims, eos="RKE", tr=0.6, nwall=0, form=form))
        b = g.memory()
        g.close()
        return b

    monkeypatch.delenv("CPMP_FUSE", raising=False)
    v1 = memory("v1", None)
    assert memory("moments", None) - v1 >= 12 * word * n
    assert memory("moments", "4") - v1 >= 12 * word * n
    assert memory("march", "4") - v1 < 12 * word * n
    assert memory(None, "4") - v1 < 12 * word * n


@pytest.mark.parametrize("form,dims,moments", [
    ("fp64", (428, 2, 225), False), ("fp64", (873, 2, 263), True), ("fp64", (496, 2, 1368), False),
    ("fp64", (922, 3, 36), False), ("fp64", (981, 3, 70), False), ("fp64", (946, 3, 298), True),
    ("fp64", (968, 4, 34), False), ("fp64", (826, 4, 70), True),
    ("fp64", (300, 5, 60), True), ("fp64", (1, 300, 400), False), ("fp64", (1, 146, 582), True),
    ("fp32a", (544, 2, 83), False), ("fp32a", (489, 2, 197), True), ("fp32a", (922, 3, 36), True),
    ("fp32", (212, 2, 1264), False), ("fp32", (562, 2, 996), True), ("fp32", (100, 2, 1067), True),
])
def test_thin_lattices_take_the_faster_path(cpmp, monkeypatch, form, dims, moments):
    """lattices of one plane or of 2 to 4 rows on both sides of the rule; the moment set, 12
    values per node and more, shows in the lattice's memory"""
    n, word = dims[0] * dims[1] * dims[2], 8 if form == "fp64" else 4

    def memory(collide):
        monkeypatch.setenv("CPMP_COLLIDE", collide) if collide else monkeypatch.delenv("CPMP_COLLIDE", raising=False)
        g = cpmp.Lattice(cpmp.make_params(*dims, eos="RKE", tr=0.6, nwall=0, form=form))
        b = g.memory()
        g.close()
        return b

    monkeypatch.delenv("CPMP_FUSE", raising=False)
    monkeypatch.delenv("CPMP_XC", raising=False)
    assert (memory(None) - memory("v1") >= 12 * word * n) == moments


# what a program does between calls: it must leave the moments usable or give them up
BETWEEN = {
    "checkpoint": lambda g, tmp: g.checkpoint_save(str(tmp / "c.ckp")),
    "plt": lambda g, tmp: g.write_plt(str(tmp / "c.plt")),
    "fields": lambda g, tmp: [g.get(k) for k in ("rho", "mu", "mv", "vel", "force", "f", "type")],
    "reduce": lambda g, tmp: g.reduce(),
    "set": lambda g, tmp: [g.set(k, g.get(k)) for k in ("f", "rho", "mu")],
    "reload": lambda g, tmp: (g.checkpoint_save(str(tmp / "r.ckp")), g.checkpoint_load(str(tmp / "r.ckp"))),
}
SETTLED = [((64, 16, 64), 4, 3, {}), ((64, 16, 64), 4, 0, {}), ((12, 13, 34), 5, 3, {}), ((20, 1, 191), 6, 3, {})]


@pytest.mark.parametrize("form", ["fp64", "fp32", "fp32a"])
@pytest.mark.parametrize("case", SETTLED, ids=lambda c: "x".join(map(str, c[0])) + "w%d" % c[2])
@pytest.mark.parametrize("what", list(BETWEEN))
def test_calls_between_runs_leave_the_run_as_it_is(cpmp, monkeypatch, tmp_path, what, case, form):
    """after one and after two steps, when the moments sit in their own buffer and in the
    population set that is not current: the same call between two runs of steps, against an
    undisturbed run, bit for bit, on tiled and other lattices; and the fields it returns
    come out the same twice"""
    a = lattice(cpmp, monkeypatch, case, form, "moments")
    b = lattice(cpmp, monkeypatch, case, form, "moments")
    for n in (1, 2, 3):
        for g in (a, b):
            g.step(n)
        BETWEEN[what](a, tmp_path)
        mv = a.get("mv")
        assert np.array_equal(mv, a.get("mv"))
        if what != "reload":        # a checkpoint does not hold MV
            assert np.array_equal(mv, b.get("mv"))
    for g in (a, b):
        g.step(2)
    for field in ("rho", "mu", "f", "mv"):
        assert np.array_equal(a.get(field), b.get(field)), field
    a.close()
    b.close()


@pytest.mark.parametrize("form", ["fp64", "fp32", "fp32a"])
def test_populations_set_between_runs_are_taken(cpmp, monkeypatch, form):
    """the state of another lattice set over moments that are current"""
    case = SETTLED[0]
    for n in (1, 2):
        a = lattice(cpmp, monkeypatch, case, form, "moments")
        b = lattice(cpmp, monkeypatch, case, form, "moments")
        a.step(n)
        b.step(5)
        for field in ("f", "rho"):
            a.set(field, b.get(field))
        a.step(3)
        b.step(3)
        for field in ("rho", "f"):
            assert np.array_equal(a.get(field), b.get(field)), field
        a.close()
        b.close()
