"""GPU: host arrays through the pinned areas.  Sizes below an area, above both areas, with
arrays that end inside an area, against the device-resident solve of the same energies
(the same kernels on the same padded blocks: equal to the bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm,nx,nE", [(32, 3, 1), (96, 7, 9), (128, 6, 40)])
def test_host_energies_equal_device_solve(nm, nx, nE):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from liteqt_amd import configs, rgf
    Hii, H1i = configs.random_device(nm, nx, 60 + nm)
    E = np.linspace(-0.4, 0.5, nE) if nE > 1 else np.array([0.1])
    sL, sG, sR = configs.scattering_self_energies(nm, nx, 61, E=E, scale=1e-2)
    p = rgf.params(rgf.MODE_COMPAT)
    got = rgf.rgf_rs_energies(p, (300.0, 300.0), E, (0.1, -0.1), Hii, H1i, sL, sG, sR)
    td = rgf.to_device_blocks
    names = ("ldos", "ndens", "pdens", "GRi1", "GLi1", "GGi1")
    out = {k: torch.zeros(nE, nx, nm, nm, dtype=torch.complex128, device="cuda") for k in names}
    out["cur"] = torch.zeros(nE, nx, nm, nm, dtype=torch.float64, device="cuda")
    out["tr"] = torch.zeros(nE, dtype=torch.float64, device="cuda")
    out["tre"] = torch.zeros(nE, dtype=torch.float64, device="cuda")
    rgf.solve_batched(p, torch.tensor(E, device="cuda"), (300.0, 300.0), (0.1, -0.1), td(Hii), td(H1i), sigL=td(sL),
                      sigR=td(sR), out=out)
    torch.cuda.synchronize()
    for k in names + ("cur",):
        assert np.array_equal(got[k], np.asarray(out[k].cpu().numpy().T)), k
    assert np.array_equal(got["tr"], out["tr"].cpu().numpy()) and np.array_equal(got["tre"], out["tre"].cpu().numpy())
