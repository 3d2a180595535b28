"""The FP64 equation-of-state part of the chemical potential on the device: its logarithm,
and every EOS, against extended precision.  Without interface energy (Ka = 0) and with
K = 1, mu of the first step is the EOS's own mu of the initial density."""
import numpy as np
import pytest

from test_gpu_production import EOS_TRS, eos_term_scale

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
DIMS = (64, 64, 64)
N = DIMS[0] * DIMS[1] * DIMS[2]


def device_mu(cpmp, rho, eos, A, B, T):
    p = cpmp.make_params(*DIMS, eos=eos, tr=0.8, nwall=0, K=1.0, Ka=0.0)
    p.A, p.B, p.T = A, B, T
    g = cpmp.Lattice(p)
    g.init_from_rho(rho)
    g.step(1)
    mu = g.get("mu")
    g.close()
    return mu


def test_logarithm(cpmp):
    """Carnahan-Starling with A = 0, T = 1 and a B of 1e-300 is the logarithm of the density.  Densities
    over the whole range of normal and subnormal numbers below the clamp at 9.7, around 1
    where the result cancels, and around the points where the reduction changes sides"""
    rng = np.random.default_rng(1)
    n = N // 4
    wide = np.ldexp(rng.uniform(0.5, 1.0, n), rng.integers(-1073, 3, n))
    near = 1 + rng.uniform(-1, 1, n) * 2.0 ** -rng.uniform(1, 52, n)
    edge = np.ldexp(np.sqrt(0.5) * (1 + rng.uniform(-1, 1, n) * 2.0 ** -rng.uniform(1, 52, n)), rng.integers(-3, 4, n))
    rho = np.concatenate([wide, near, edge, rng.uniform(1e-3, 9.7, N - 3 * n)])
    rho = np.where(rho > 9.7, 9.7, np.where(rho == 1.0, 0.5, rho))
    rho[:3] = 0.0, 5e-324, 1.0
    mu = device_mu(cpmp, rho, "CSE", 0.0, 1e-300, 1.0)
    assert mu[0] == -np.inf and abs(mu[2]) < 1e-298
    mu, rho = np.delete(mu, [0, 2]), np.delete(rho, [0, 2])
    ref = np.log(rho.astype(np.longdouble))
    ulp = np.spacing(np.maximum(np.abs(ref.astype(np.float64)), np.finfo(float).tiny))
    err = float(np.max(np.abs(mu - ref) / ulp))
    print(f"[eos] logarithm: {err:.3f} ulp", flush=True)
    assert err < 0.6


def mu_extended(eos, A, B, T, d):
    """the closed forms in extended precision"""
    A, B, T, d = (np.asarray(v, np.longdouble) for v in (A, B, T, d))
    d = np.where(d > 9.7, np.longdouble(9.7) + (d - np.longdouble(9.7)) / (1 + (d - np.longdouble(9.7)) * 1.5), d)
    bd, om, s2 = B * d, 1 - B * d, np.sqrt(np.longdouble(2))
    if eos in ("PRW", "PRM"):
        return (T * np.log(d / om) - A / (2 * s2 * B) * np.log((s2 - 1 + bd) / (s2 + 1 - bd)) + T / om
                - A * d / (1 + 2 * bd - bd * bd)), d
    if eos == "VDW":
        return T * np.log(d / om) + T / om - 2 * A * d, d
    if eos in ("RKE", "RKS"):
        return T * np.log(d / om) + T / om - A / B * np.log(1 + bd) - A * d / (1 + bd), d
    return T * (np.log(d) + (8 * bd - 9 * bd * bd + 3 * bd ** 3) / om ** 3) - 2 * A * d, d


@pytest.mark.parametrize("eos,tr", EOS_TRS)
def test_every_eos(cpmp, eos, tr):
    """Each term carries at most 16 roundings of its size (the reciprocal and its products, a
    cube, a logarithm of an argument that is off by as many), and the rounding of b d enters
    1 - b d magnified by b d / (1 - b d), three times in the cube; the argument of a logarithm
    errs against 1, not against the logarithm."""
    A, B, Tc, Rc = cpmp.set_multiphase(eos, tr)
    T = tr * Tc
    top = min(12.0, 0.98 / B)
    rho = np.exp(np.random.default_rng(2).uniform(np.log(1e-4 * top), np.log(top), N))
    mu = device_mu(cpmp, rho, eos, A, B, T)
    ref, d = mu_extended(eos, A, B, T, rho)
    d = d.astype(np.float64)
    om = 1 - B * d
    scale = eos_term_scale(eos, A, B, T, d) + T + A / B
    bound = U * scale * (16 + 3 * B * d / om)
    ratio = float(np.max(np.abs(mu - ref) / bound))
    print(f"[eos] {eos}: {ratio:.3f} of the bound", flush=True)
    assert ratio < 1


@pytest.mark.parametrize("eos", [e for e, _ in EOS_TRS])
def test_limits(cpmp, eos):
    """the densest packing, b d = 1, an empty node, and densities far past the clamp keep the
    values of the closed forms"""
    rho = np.full(N, 4.0)
    assert np.all(device_mu(cpmp, rho, eos, 1.0, 0.25, 1.0) == np.inf)
    rho[:] = 0.0
    assert np.all(device_mu(cpmp, rho, eos, 1.0, 0.0625, 1.0) == -np.inf)
    rho[:] = 1e300
    ref, _ = mu_extended(eos, 1.0, 0.0625, 1.0, 1e300)
    assert np.all(np.abs(device_mu(cpmp, rho, eos, 1.0, 0.0625, 1.0) - np.float64(ref)) < 1e-13)
