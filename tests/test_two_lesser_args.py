"""CPU: the second lesser source's arguments are checked before anything runs: its blocks have
the batch's energy stride, and the plain path does not take one."""
import pytest
import torch

from liteqt_amd import rgf

NM, NX, NE = 32, 3, 4


def _args(per_energy):
    c = lambda *s: torch.zeros(*s, dtype=torch.complex128)
    blk = (NE, NX, NM, NM) if per_energy else (NX, NM, NM)
    return dict(E=torch.zeros(NE, dtype=torch.float64), temp=(300.0, 300.0), mu=(0.0, 0.0), Hii=c(NX, NM, NM),
                H1i=c(NX, NM, NM), sigL=c(*blk), sigR=c(*blk)), c(NE, NX, NM, NM)


@pytest.mark.parametrize("name", ["sigL", "sigL_up"])
@pytest.mark.parametrize("per_energy", [False, True])
def test_second_source_of_another_stride_is_refused(name, per_energy):
    kw, nd = _args(per_energy)
    other = torch.zeros(*((NX, NM, NM) if per_energy else (NE, NX, NM, NM)), dtype=torch.complex128)
    with pytest.raises(rgf.RgfError, match="second"):
        rgf.solve_batched(rgf.params(rgf.MODE_PHYSICAL), second={name: other, "ndens": nd}, **kw)


def test_plain_path_refuses_a_second_source():
    kw, nd = _args(True)
    with pytest.raises(rgf.RgfError, match="plain path takes one"):
        rgf.solve_batched(rgf.params(rgf.MODE_PHYSICAL), second={"ndens": nd}, plain=True, **kw)
