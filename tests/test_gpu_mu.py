"""The two chemical-potential kernels of the FP32-storage forms, by columns and as a march
over 8 x 32 tiles (large lattices), run the same arithmetic per node: the same bits."""
import numpy as np
import pytest

import gpu_cases as gc

pytestmark = pytest.mark.gpu

# dims, planes per workgroup, walls, Laplacian points: edges of the tiles and chunks, fewer
# planes than the stencil reaches, odd and even chunk lengths
CASES = [((1, 8, 32), 8, 0, 5), ((5, 9, 33), 3, 3, 7), ((7, 7, 31), 32, 0, 7), ((9, 1, 65), 4, 3, 5),
         ((16, 16, 64), 8, 3, 5), ((33, 25, 70), 16, 0, 5), ((12, 3, 2), 1, 0, 7)]


def lattice(cpmp, monkeypatch, case, form, kernel):
    dims, xc, nwall, lap = case
    monkeypatch.setenv("CPMP_MU", kernel)
    monkeypatch.setenv("CPMP_COLLIDE", "v1")
    monkeypatch.setenv("CPMP_XC", str(xc))
    dg, dl = gc.densities("RKE", 0.60)
    g = cpmp.Lattice(cpmp.make_params(*dims, eos="RKE", tr=0.6, nwall=nwall, form=form, lap_points=lap))
    for v in ("CPMP_MU", "CPMP_COLLIDE", "CPMP_XC"):
        monkeypatch.delenv(v)
    g.set_wall_mu(-0.01, 0.02)
    # gas, liquid and interface nodes side by side: both branches of the EOS in every wave
    rho = np.random.default_rng(5).uniform(dg, dl, dims)
    rho[:, :, :nwall] = rho[:, :, dims[2] - nwall:] = 0
    g.init_from_rho(rho.ravel())
    return g, rho.ravel()


@pytest.mark.parametrize("form", ["fp32", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0])))
def test_march_and_columns_give_the_same_bits(cpmp, monkeypatch, case, form):
    res = []
    for kernel in ("columns", "march"):
        g, _ = lattice(cpmp, monkeypatch, case, form, kernel)
        first = []
        for _ in range(2):
            g.step(1)
            first += [g.get("mu"), g.get("rho")]
        res.append(first)
        g.close()
    for a, b in zip(*res):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.isfinite(res[0][0]).all()


def test_march_records_the_tape_of_the_adjoint(cpmp, monkeypatch):
    res = []
    for kernel in ("columns", "march"):
        g, rho = lattice(cpmp, monkeypatch, ((12, 9, 40), 5, 3, 5), "fp32", kernel)
        # a smooth field: the mean of gas and liquid with a tenth of the noise
        rho = np.where(rho > 0, 4.0 + 0.1 * (rho - 4.0), 0.0)
        g.init_from_rho(rho)
        res.append(g.adjoint(4, rho * 1.01, checkpoint_every=2))
        g.close()
    a, b = res
    assert a[0] == b[0] and a[3] == b[3] and np.isfinite(a[0])
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
