"""GPU: an energy solved by a group of workgroups (blocks of 64 to 256 orbitals, few
energies; at 32 orbitals a second workgroup for the right contact) against the one-workgroup solve of the same energy, which a caller's slot limit
selects.  Both form every output element from the same products in the same order; the
bound is the rounding of one reordering, n eps times the conditioning at eta = 1e-3
(256 * 1.1e-16 * 1e2 < 1e-11), relative per output array."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _env():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from liteqt_amd import configs, rgf
    return torch, configs, rgf


def _device(nm, nx, nE, seed):
    torch, configs, rgf = _env()
    Hii, H1i = configs.random_device(nm, nx, seed)
    E = torch.tensor(np.linspace(-0.6, 0.7, nE) if nE > 1 else np.array([0.1]), dtype=torch.float64, device="cuda")
    return torch, configs, rgf, rgf.to_device_blocks(Hii), rgf.to_device_blocks(H1i), E


def _close(a, b, name):
    d = (a - b).norm() / b.norm()
    assert d <= TOL, (name, float(d))


# one energy takes the largest group, 9 energies two groups an XCD, 40 the smallest tiles
# per rank with every variant of the inverse; 300 leaves a tail of 44 behind a full round; 32
# orbitals in pairs, 128 energies the most
@pytest.mark.parametrize("nm,nE", [(96, 1), (96, 40), (128, 1), (128, 9), (160, 3), (192, 9), (224, 1), (256, 1), (256, 17),
                                   (96, 300), (32, 1), (32, 128), (64, 1), (64, 9)])
@pytest.mark.parametrize("mode", ["compat", "physical"])
def test_group_solve_equals_one_workgroup(nm, nE, mode):
    torch, configs, rgf, H, C, E = _device(nm, 4, nE, 10 + nm)
    p = rgf.params(rgf.MODE_COMPAT if mode == "compat" else rgf.MODE_PHYSICAL, eta_dev=1e-3)
    nx = 4
    sl, _, sr = configs.scattering_self_energies(nm, nx, 3, E=0.1, scale=1e-2)
    sig = {} if nE == 9 else {"sigL": rgf.to_device_blocks(sl), "sigR": rgf.to_device_blocks(sr)}
    res = []
    for slots in (0, nE):
        blk = lambda dt: torch.zeros(nE, nx, nm, nm, dtype=dt, device="cuda")
        out = {k: blk(torch.complex128) for k in ("ldos", "ndens", "pdens", "GRi1", "GLi1", "GGi1")}
        out["cur"] = blk(torch.float64)
        for k in ("tr", "tre"):
            out[k] = torch.zeros(nE, dtype=torch.float64, device="cuda")
        for k in ("dens_n", "dens_p"):
            out[k] = torch.zeros(nE, nx, dtype=torch.float64, device="cuda")
        out["info"] = torch.zeros(nE, 4, dtype=torch.int32, device="cuda")
        rgf.solve_batched(p, E, (300.0, 300.0), (0.1, -0.1), H, C, out=out, max_slots=slots, **sig)
        torch.cuda.synchronize()
        res.append(out)
    assert torch.equal(res[0]["info"], res[1]["info"])
    for k in res[0]:
        if k != "info":
            _close(res[0][k], res[1][k], k)


@pytest.mark.parametrize("nm,nE", [(96, 5), (128, 3), (256, 2)])
def test_group_offdiag_refresh_equals_one_workgroup(nm, nE):
    nx = 4
    torch, configs, rgf, H, C, E = _device(nm, nx, nE, 20 + nm)
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3)
    names = ("sigL", "sigR", "sigR_lo", "sigR_up", "sigL_up")
    blocks = configs.offdiag_self_energies(configs.scattering_blocks(nm, nx, 4, scale=1e-2), 0.4)
    res = []
    for slots in (0, nE):
        sig = {k: rgf.to_device_blocks(b).unsqueeze(0).repeat(nE, 1, 1, 1).contiguous() for k, b in zip(names, blocks)}
        out = {"tr": torch.zeros(nE, dtype=torch.float64, device="cuda"),
               "dens_p": torch.zeros(nE, nx, dtype=torch.float64, device="cuda")}
        rgf.solve_batched(p, E, (300.0, 300.0), (0.1, -0.1), H, C, out=out, max_slots=slots, scba=(1e-2, 0.5), **sig)
        torch.cuda.synchronize()
        res.append({**out, **sig})
    for k in res[0]:
        _close(res[0][k], res[1][k], k)


@pytest.mark.parametrize("nm,nE,ckpt", [(96, 4, 0), (128, 100, 0), (256, 3, 0), (128, 3, 2)])
def test_group_adjoint_equals_one_workgroup(nm, nE, ckpt):
    nx = 5
    torch, configs, rgf, H, C, E = _device(nm, nx, nE, 30 + nm)
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3)
    g = torch.Generator(device="cuda").manual_seed(1)
    w_tr = torch.rand(nE, dtype=torch.float64, device="cuda", generator=g)
    w_n = torch.rand(nE, nx, dtype=torch.float64, device="cuda", generator=g)
    res = [rgf.adjoint_batched(p, E, (300.0, 300.0), (0.1, -0.1), H, C, w_tr=w_tr, w_n=w_n, max_slots=slots, ckpt=ckpt)
           for slots in (0, nE)]
    torch.cuda.synchronize()
    for a, b, name in zip(res[0], res[1], ("J", "dU", "dH")):
        _close(a, b, name)


# the screened interaction has no slot limit: 3 energies alone (groups) against the same
# energies as the first of 256 (one workgroup each)
@pytest.mark.parametrize("nm", [96, 128, 200])
def test_group_w_equals_one_workgroup(nm):
    torch, configs, rgf = _env()
    nx, nE = 4, 3
    g = torch.Generator(device="cuda").manual_seed(nm)
    cn = lambda *s: torch.randn(*s, dtype=torch.complex128, device="cuda", generator=g) / nm ** 0.5
    V, V1, P = cn(nx, nm, nm), cn(nx, nm, nm) * 0.3, [cn(nE, nx, nm, nm) * 0.2 for _ in range(3)]
    few = rgf.w_solve_batched(V, V1, *P, want_i1=True)
    many = rgf.w_solve_batched(V, V1, *[torch.cat([x, x[:1].expand(256 - nE, -1, -1, -1)]).contiguous() for x in P],
                               want_i1=True)
    torch.cuda.synchronize()
    for k in ("WL", "WG", "WR", "WRi1"):
        _close(few[k], many[k][:nE], k)
    assert int(few["info"].sum()) == 0


def test_group_singular_slab_is_zeroed_and_counted():
    """A singular slab block (above and below 128 orbitals) is zeroed and counted once by a group, as by one workgroup."""
    for nm in (128, 160):
        nx, nE = 3, 2
        torch, configs, rgf, H, C, E = _device(nm, nx, nE, 40 + nm)
        H, C = torch.zeros_like(H), torch.zeros_like(C)
        E = torch.zeros_like(E)
        p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=0.0)
        res = []
        for slots in (0, nE):
            out = {"ldos": torch.full((nE, nx, nm, nm), 7.0, dtype=torch.complex128, device="cuda"),
                   "info": torch.zeros(nE, 4, dtype=torch.int32, device="cuda")}
            rgf.solve_batched(p, E, (300.0, 300.0), (0.0, 0.0), H, C, out=out, max_slots=slots)
            torch.cuda.synchronize()
            res.append(out)
        assert torch.equal(res[0]["info"], res[1]["info"]) and int(res[0]["info"][0, 3]) == nx
        assert torch.equal(res[0]["ldos"], res[1]["ldos"]) and float(res[0]["ldos"].abs().max()) == 0.0


# block sizes of every kind of group (32 and 64 on one workgroup, lists of several items),
# fewer and more items than the 256 compute units
@pytest.mark.parametrize("counts", [(3, 2, 5, 2, 1, 2, 1), (200, 40, 9, 7, 3, 2, 4)])
def test_group_devices_equal_one_workgroup(counts):
    torch, configs, rgf = _env()
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3)
    devs, ref = [], []
    for j, (nm, nE) in enumerate(zip((32, 64, 96, 128, 160, 192, 256), counts)):
        nx = 3 + j % 3
        _, _, _, H, C, E = _device(nm, nx, nE, 50 + nm)
        new = lambda: {"tr": torch.zeros(nE, dtype=torch.float64, device="cuda"),
                       "dens_n": torch.zeros(nE, nx, dtype=torch.float64, device="cuda"),
                       "info": torch.zeros(nE, 4, dtype=torch.int32, device="cuda")}
        devs.append({"E": E, "temp": (300.0, 300.0), "mu": (0.1, -0.1), "Hii": H, "H1i": C, "out": new()})
        ref.append(rgf.solve_batched(p, E, (300.0, 300.0), (0.1, -0.1), H, C, out=new(), max_slots=nE))
    _, rep = rgf.solve_devices(p, devs)
    torch.cuda.synchronize()
    assert rep["items"] == sum(counts)
    for d, r in zip(devs, ref):
        assert torch.equal(d["out"]["info"], r["info"])
        _close(d["out"]["tr"], r["tr"], "tr")
        _close(d["out"]["dens_n"], r["dens_n"], "dens_n")


def _decimation_sum(nm, nE):
    """The left contact's sum of |C_ij| after one iteration, to the bit, as each of nE equal
    energies forms it: the smallest tolerance that it passes."""
    torch, configs, rgf, H, C, _ = _device(nm, 2, 1, 10 + nm)
    E = torch.full((nE,), 0.1, dtype=torch.float64, device="cuda")
    info = torch.zeros(nE, 4, dtype=torch.int32, device="cuda")
    lo, hi = np.zeros(nE, np.int64), np.full(nE, np.float64(1e30).view(np.int64))  # fails, passes
    while (hi - lo).max() > 1:
        mid = lo + (hi - lo) // 2  # (the sum of two such patterns passes 63 bits)
        e = int((hi - lo).argmax())
        rgf.solve_batched(rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3, dec_nmax=1, dec_tol=float(mid[e:e + 1].view(np.float64)[0])),
                          E, (300.0, 300.0), (0.1, -0.1), H, C, out={"info": info})
        passed = (info[:, 2].cpu().numpy() & 1) == 0
        hi = np.where(passed & (mid[e] < hi), mid[e], hi)
        lo = np.where(~passed & (mid[e] > lo), mid[e], lo)
    return hi


# groups whose GEMMs take 32 x 32 tiles (one energy, 16 or 32 ranks) and 128 x 64 tiles (many
# energies, 2 or 4 ranks): the sum that ends the decimation is the same, to the bit
@pytest.mark.parametrize("nm,many", [(128, 128), (256, 64)])
def test_decimation_sum_does_not_depend_on_the_group(nm, many):
    one, sums = _decimation_sum(nm, 1), _decimation_sum(nm, many)
    assert (sums == one[0]).all(), (one[:1].view(np.float64), sums.view(np.float64))


# one item takes a group of up to 16 workgroups (32 x 32 tiles), 128 of them one of two each
# (128 x 64), 257 energies of 32 orbitals the work list with its variants
@pytest.mark.parametrize("nm,nE,groups,tile", [(128, 1, True, 1), (128, 128, True, 4), (32, 257, False, 1)])
def test_devices_report_what_runs(nm, nE, groups, tile):
    torch, configs, rgf, H, C, E = _device(nm, 4, nE, 10 + nm)
    dev = {"E": E, "temp": (300.0, 300.0), "mu": (0.1, -0.1), "Hii": H, "H1i": C,
           "out": {"tr": torch.zeros(nE, dtype=torch.float64, device="cuda")}}
    tiles, rep = rgf.solve_devices(rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3), [dev], autotune=groups)
    torch.cuda.synchronize()
    assert tiles == [tile] and rep["items"] == nE
    if groups:
        assert rep["slots"] > nE and rep["tuned"] == 0
    else:
        assert rep["slots"] <= nE


# full rounds of one energy per workgroup, then groups on the same slots (256 + 4 energies), and
# 64 orbitals, where every rank sweeps the whole block
@pytest.mark.parametrize("nm,nE", [(96, 260), (64, 9)])
def test_group_adjoint_behind_full_rounds(nm, nE):
    test_group_adjoint_equals_one_workgroup(nm, nE, 0)


@pytest.mark.parametrize("nm,nE", [(96, 260), (64, 9)])
def test_group_offdiag_refresh_behind_full_rounds(nm, nE):
    test_group_offdiag_refresh_equals_one_workgroup(nm, nE)


# (the W solve's one-workgroup form: as the first of 256 energies)
@pytest.mark.parametrize("nm,nE", [(96, 260), (64, 3)])
def test_group_w_behind_full_rounds(nm, nE):
    torch, configs, rgf = _env()
    nx = 3
    g = torch.Generator(device="cuda").manual_seed(nm)
    cn = lambda *s: torch.randn(*s, dtype=torch.complex128, device="cuda", generator=g) / nm ** 0.5
    V, V1, P = cn(nx, nm, nm), cn(nx, nm, nm) * 0.3, [cn(nE, nx, nm, nm) * 0.2 for _ in range(3)]
    got = rgf.w_solve_batched(V, V1, *P)
    tail = nE % 256
    lone = rgf.w_solve_batched(V, V1, *[torch.cat([x[nE - tail:], x[:1].expand(256 - tail, -1, -1, -1)]).contiguous() for x in P])
    rest = rgf.w_solve_batched(V, V1, *[x[:256].contiguous() for x in P]) if nE > 256 else None
    torch.cuda.synchronize()
    for k in ("WL", "WG", "WR"):
        _close(got[k][nE - tail:], lone[k][:tail], k)
        if rest:
            assert torch.equal(got[k][:256], rest[k]), k
    assert int(got["info"].sum()) == 0


def test_group_singular_slab_at_64_orbitals():
    nm, nx, nE = 64, 3, 2
    torch, configs, rgf, H, C, E = _device(nm, nx, nE, 40 + nm)
    H, C, E = torch.zeros_like(H), torch.zeros_like(C), torch.zeros_like(E)
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=0.0)
    for slots in (0, nE):
        out = {"ldos": torch.full((nE, nx, nm, nm), 7.0, dtype=torch.complex128, device="cuda"),
               "info": torch.zeros(nE, 4, dtype=torch.int32, device="cuda")}
        rgf.solve_batched(p, E, (300.0, 300.0), (0.0, 0.0), H, C, out=out, max_slots=slots)
        torch.cuda.synchronize()
        assert int(out["info"][:, 3].min()) == int(out["info"][:, 3].max()) == nx
        assert float(out["ldos"].abs().max()) == 0.0
