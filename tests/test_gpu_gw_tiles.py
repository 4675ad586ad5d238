"""Band elements of the GW step at the edges of its tiles (256 outputs, steps in blocks of
16, one to sixteen waves) and with the off-band elements in the same launch, against the
oracle.  Tolerance: a sum of n <= 3072 random products of FP64 numbers is off by at most
n * 1.1e-16 * sqrt(n) ~ 2e-11 of its norm; 1e-10 of the largest output of the step."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from liteqt_amd import gw
from oracle import gw_oracle as orc

pytestmark = pytest.mark.gpu


def _rand(rng, shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("nm,nx,nen,ndiag,nopmax", [
    (2, 5, 2, 0, 0), (3, 5, 17, 1, 7), (9, 5, 256, 1, 127), (5, 6, 257, 2, 16), (4, 5, 514, 1, 255),
    (4, 5, 515, 1, 256), (3, 5, 1030, 1, 514), (2, 5, 1744, 0, 871), (2, 5, 2040, 1, 1019),
    (12, 5, 70, 8, 20), (2, 5, 3072, 1, 1535)])
def test_band_tiles(nm, nx, nen, ndiag, nopmax):
    print(f"gw tiles nm={nm} nx={nx} nen={nen} ndiag={ndiag} nopmax={nopmax}", flush=True)
    rng = np.random.default_rng(nen)
    G, W, S = ([_rand(rng, (nm, nm, nx, nen)) for _ in range(3)] for _ in range(3))
    dE_P, dE_S = 0.3 - 0.2j, 0.1 + 0.4j
    p = gw.params(nm, nx, nen, ndiag, nopmax, dE_P, dE_S, 0.6)
    g = [gw.to_device(a) for a in G]
    P = [torch.full((nen, nx, nm, nm), float("nan"), dtype=torch.complex128, device="cuda:0") for _ in range(3)]
    gw.polarization(p, *g, *P)
    s = [gw.to_device(a) for a in S]
    gw.selfenergy(p, *g, *[gw.to_device(a) for a in W], *s)
    torch.cuda.synchronize()
    for got, want in ((P, orc.polarization(*G, ndiag, nopmax, dE_P)),
                      (s, orc.selfenergy_step(*G, *W, *S, ndiag, nopmax, dE_S, 0.6))):
        scale = max(np.linalg.norm(r) for r in want)  # P^r of a diagonal at nop = 0 is zero
        for t, ref in zip(got, want):
            assert np.linalg.norm(gw.to_host(t) - ref) <= 1e-10 * scale
