"""GPU: calls on several streams share the engine's workspace.  Each call's outputs equal
those of the same call by itself, to the bit (the same kernels on the same inputs), also
where the calls' work would overlap on the device; and a call captured into a graph of the
caller's gives the eager results on every replay."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T, MU = (300.0, 300.0), (0.1, -0.1)


def _env():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible")
    from liteqt_amd import configs, rgf
    return torch, configs, rgf


def _solve(torch, configs, rgf, nm, nx, nE):
    """A solve of nE energies: a function of the output tensors, and a maker of those."""
    Hii, H1i = configs.random_device(nm, nx, 70 + nm)
    H, C = rgf.to_device_blocks(Hii), rgf.to_device_blocks(H1i)
    E = torch.tensor(np.linspace(-0.6, 0.7, nE), dtype=torch.float64, device="cuda")
    p = rgf.params(rgf.MODE_PHYSICAL, eta_dev=1e-3)

    def new():
        return {"ldos": torch.zeros(nE, nx, nm, nm, dtype=torch.complex128, device="cuda"),
                "tr": torch.zeros(nE, dtype=torch.float64, device="cuda"),
                "info": torch.zeros(nE, 4, dtype=torch.int32, device="cuda")}

    return (lambda out, **kw: rgf.solve_batched(p, E, T, MU, H, C, out=out, **kw)), new, (p, E, H, C)


# groups of several sizes, pairs and lone workgroups, solve, adjoint and W, alternating
# between two streams
def test_calls_on_two_streams_do_not_meet_in_the_workspace():
    torch, configs, rgf = _env()
    jobs = [_solve(torch, configs, rgf, nm, nx, nE)
            for nm, nx, nE in ((128, 12, 9), (96, 4, 20), (32, 6, 40), (64, 5, 3), (128, 3, 300), (256, 3, 2))]
    ref = []
    for run, new, _ in jobs:
        ref.append(new())
        run(ref[-1])
        torch.cuda.synchronize()
    p, E, H, C = jobs[0][2]
    adj = lambda: rgf.adjoint_batched(p, E, T, MU, H, C, w_tr=torch.ones_like(E))
    adj_ref = [x.clone() for x in adj()]
    g = torch.Generator(device="cuda").manual_seed(3)
    cn = lambda *s: torch.randn(*s, dtype=torch.complex128, device="cuda", generator=g) / 96 ** 0.5
    w_in = (cn(4, 96, 96), cn(4, 96, 96) * 0.3, *[cn(5, 4, 96, 96) * 0.2 for _ in range(3)])
    w_ref = {k: v.clone() for k, v in rgf.w_solve_batched(*w_in).items() if v is not None}
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got, k = [], 0
    for rounds in range(3):
        print("two streams, round", rounds, flush=True)
        for run, new, _ in jobs:
            out = new()
            torch.cuda.current_stream().synchronize()
            with torch.cuda.stream(streams[k % 2]):
                run(out)
            got.append(out)
            k += 1
        with torch.cuda.stream(streams[k % 2]):
            a = adj()
        with torch.cuda.stream(streams[(k + 1) % 2]):
            w = rgf.w_solve_batched(*w_in)
        k += 1
        torch.cuda.synchronize()
        for x, y in zip(a, adj_ref):
            assert torch.equal(x, y)
        for n in w_ref:
            assert torch.equal(w[n], w_ref[n]), n
    for i, out in enumerate(got):
        for n in out:
            assert torch.equal(out[n], ref[i % len(jobs)][n]), (i, n)


# few energies (eager: groups; captured: one workgroup per energy), replayed with eager
# calls in between
def test_captured_call_equals_eager_on_every_replay():
    torch, configs, rgf = _env()
    run, new, _ = _solve(torch, configs, rgf, 96, 4, 6)
    other, other_new, _ = _solve(torch, configs, rgf, 128, 3, 5)
    ref, out, o = new(), new(), other_new()
    run(ref, max_slots=6)
    run(new())
    other(o)
    torch.cuda.synchronize()
    want = o["ldos"].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(out)
    for rep in range(3):
        print("captured call, replay", rep, flush=True)
        for v in out.values():
            v.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for n in ref:
            assert torch.equal(out[n], ref[n]), (rep, n)
        other(o)
        torch.cuda.synchronize()
        assert torch.equal(o["ldos"], want)
