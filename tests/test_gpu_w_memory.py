"""GPU: device memory of the screened interaction by super-blocks (gw.w_blocks).  A chunk
holds at its peak at most 13.1 arrays of its super-blocks, which is what it took with one
lesser source per solve (13.15 to 13.4 measured; the arrays are the three of Sigma^R, X and
its two off-diagonals, and the two sources with their temporaries)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nm,nx,nE", [(64, 9, 40), (16, 6, 300), (32, 1, 100)])
def test_w_blocks_peak_memory(nm, nx, nE):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from liteqt_amd import gw
    g = torch.Generator(device="cuda").manual_seed(1)
    cn = lambda *s: torch.randn(*s, dtype=torch.complex128, device="cuda", generator=g) / nm ** 0.5
    V, V1, PR = cn(nx, nm, nm), cn(nx, nm, nm) * 0.3, cn(nE, nx, nm, nm) * 0.2
    anti = lambda a: (a - a.conj().transpose(-1, -2)).contiguous()
    PL, PG = (anti(cn(nE, nx, nm, nm) * 0.2) for _ in range(2))
    W = [torch.empty_like(PR) for _ in range(3)]
    gw.w_blocks(V, V1, PL, PG, PR, *W)  # library workspaces and the matrix products' own
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    gw.w_blocks(V, V1, PL, PG, PR, *W)
    torch.cuda.synchronize()
    chunk = min(nE, 256) * max(2, (nx + 1) // 2) * (2 * nm) ** 2 * 16
    assert torch.cuda.max_memory_allocated() - base <= 13.1 * chunk
