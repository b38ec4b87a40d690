"""MHDAdjoint built under one torch stream and used under another: the device's stream is ordered after the
work of the constructor's stream, which may still write the memory that the runner's buffers were handed, and
the gradients are those of a run on one stream, bit for bit."""
import numpy as np
import pytest

from astaroth_amd import astaroth as ac

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", params=["fp32", "fp64"])
def lib(request, require_gpu):
    return ac.load(request.param)


def info_of(lib):
    # the direct kernel pinned, so that the runs do not differ in what an autotuner picks
    return lib.config((20, 17, 13), AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3,
                      AC_eta=5e-3, AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True,
                      AC_solve_tile_x=-1)


def gradient(runner, f):
    from astaroth_amd import adjoint as AD
    nu, eta = (torch.tensor(5e-3, dtype=torch.float64, requires_grad=True) for _ in range(2))
    f0 = f.clone().requires_grad_(True)
    out = AD.MHDSolve.apply(f0, nu, eta, runner)
    g = torch.autograd.grad((out * out).sum(), (f0, nu, eta))
    return [out.detach()] + list(g)


def test_constructor_orders_the_device_after_its_stream(lib, monkeypatch):
    from astaroth_amd import adjoint as AD
    print(f"case runner constructor order {lib.precision}", flush=True)
    entered = []
    enter = AD.MHDAdjoint._enter

    def recorded(self):
        entered.append((torch.cuda.current_stream(self.tdev), hasattr(self, "workspace") and hasattr(self, "param_grad")))
        enter(self)

    monkeypatch.setattr(AD.MHDAdjoint, "_enter", recorded)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        runner = AD.MHDAdjoint(lib, info_of(lib), 2, 1e-3, snaps=1)
    # after both buffers were allocated, and param_grad zeroed, on that stream
    assert entered == [(side, True)]
    torch.cuda.synchronize()
    runner.close()


@pytest.mark.parametrize("schedule", ["revolve", "uniform"])
def test_built_and_used_under_two_streams(lib, schedule):
    from astaroth_amd import adjoint as AD
    print(f"case runner streams {lib.precision} {schedule}", flush=True)
    make = lambda: AD.MHDAdjoint(lib, info_of(lib), 3, 1e-3, schedule=schedule, snaps=1, every=2)  # noqa: E731
    runner = make()
    gen = torch.Generator(device="cpu").manual_seed(3)
    f = (0.02 * torch.randn(runner.shape, generator=gen, dtype=torch.float64)).to(runner.tdtype).cuda()
    torch.cuda.synchronize()
    want = [t.cpu().numpy() for t in gradient(runner, f)]
    nbytes = runner.workspace.numel()
    torch.cuda.synchronize()
    runner.close()
    del runner
    build, use = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(build):
        # the workspace's memory, handed back with the work that writes it still queued
        big = torch.ones((4096, 4096), device="cuda")
        old = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        for _ in range(20):
            big = torch.sin(big @ big)
        old.fill_(255)
        del old
        runner = make()
    with torch.cuda.stream(use):
        use.wait_stream(torch.cuda.default_stream())  # f's stream
        got = gradient(runner, f)
        got = [t.cpu().numpy() for t in got]
    torch.cuda.synchronize()
    runner.close()
    for a, b in zip(want, got):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
