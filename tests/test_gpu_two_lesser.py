"""GPU: a second lesser source carried through a block-tridiagonal-Sigma solve against a solve
of its own, which forms its G^< from the same products (bound as for a reordering: 1e-11
relative at eta = 1e-3).  3 energies of 96 orbitals run on groups of workgroups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm,nE,nx", [(32, 5, 4), (64, 3, 3), (96, 3, 4), (128, 140, 2), (160, 2, 3)])
def test_second_source_equals_its_own_solve(nm, nE, nx):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from liteqt_amd import configs, rgf
    Hii, H1i = configs.random_device(nm, nx, nm)
    H, C = rgf.to_device_blocks(Hii), rgf.to_device_blocks(H1i)
    E = torch.tensor(np.linspace(-0.6, 0.7, nE), dtype=torch.float64, device="cuda")
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3)
    names = ("sigL", "sigR", "sigR_lo", "sigR_up", "sigL_up")
    blocks = configs.offdiag_self_energies(configs.scattering_blocks(nm, nx, 4, scale=1e-2), 0.4)
    sig = {k: rgf.to_device_blocks(b).unsqueeze(0).repeat(nE, 1, 1, 1).contiguous() for k, b in zip(names, blocks)}
    other = {k: (0.3 * (1 + torch.arange(nE, device="cuda")).reshape(-1, 1, 1, 1) / nE) * sig[k] for k in ("sigL", "sigL_up")}
    new = lambda: torch.zeros(nE, nx, nm, nm, dtype=torch.complex128, device="cuda")
    T, mu = (300.0, 300.0), (0.1, -0.1)
    both, second = {"ndens": new(), "ldos": new()}, new()
    rgf.solve_batched(p, E, T, mu, H, C, out=both, second={**other, "ndens": second}, **sig)
    one, two = {"ndens": new(), "ldos": new()}, {"ndens": new()}
    rgf.solve_batched(p, E, T, mu, H, C, out=one, **sig)
    rgf.solve_batched(p, E, T, mu, H, C, out=two, **{**sig, **other})
    torch.cuda.synchronize()
    for got, ref in ((both["ndens"], one["ndens"]), (both["ldos"], one["ldos"]), (second, two["ndens"])):
        assert (got - ref).norm() <= 1e-11 * ref.norm()


def test_second_source_alone_per_energy():
    """The batch has no Sigma, the second source one per energy: each energy takes its own."""
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from liteqt_amd import configs, rgf
    nm, nE, nx = 32, 4, 3
    Hii, H1i = configs.random_device(nm, nx, nm)
    H, C = rgf.to_device_blocks(Hii), rgf.to_device_blocks(H1i)
    E = torch.tensor(np.linspace(-0.6, 0.7, nE), dtype=torch.float64, device="cuda")
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3)
    sl, _, _ = configs.scattering_self_energies(nm, nx, 4, E=np.linspace(0.0, 0.4, nE), scale=1e-2)
    sl = rgf.to_device_blocks(sl)
    new = lambda: torch.zeros(nE, nx, nm, nm, dtype=torch.complex128, device="cuda")
    second, own = new(), new()
    rgf.solve_batched(p, E, (300.0, 300.0), (0.1, -0.1), H, C, out={"ndens": new()}, second={"sigL": sl, "ndens": second})
    rgf.solve_batched(p, E, (300.0, 300.0), (0.1, -0.1), H, C, sigL=sl, out={"ndens": own})
    torch.cuda.synchronize()
    assert (second - own).norm() <= 1e-11 * own.norm()
