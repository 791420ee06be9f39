"""ELASTIC2 and EM2 on regions (several time steps per launch, the default of
all but the largest plans): whole states and receiver samples bit-identical to
the one-step kernel on 4 x 32 tiles, over grids smaller than a region, slabs of
every width, sources and receivers on the rings, shared cells, odd runs, graph
blocks, segments and mode switches; and the same unstable step."""
import numpy as np
import pytest
import torch

from helpers import tiny_problem

pytestmark = pytest.mark.gpu


def _walk(p, precision):
    from seidart_amd.solver import Simulation
    s = Simulation(p, precision=precision)
    s.use((1, 4, 32, 0))
    return s


def _same(a, b):
    torch.cuda.synchronize()
    for (_, _, x), (_, _, y) in zip(a.shots, b.shots):
        assert torch.equal(x["state"], y["state"])
        assert torch.equal(x["trace"], y["trace"])


def _ring(p):
    """Receivers on the corners and rings, on the source and twice on one cell."""
    for sh in p.shots:
        i, _, k = sh.src
        pts = [(0, 0), (p.nx - 1, p.nz - 1), (1, p.nz - 2), (p.nx - 2, 1), (i, k), (i, k), (i - 1, k), (p.nx // 2, k)]
        sh.rec = np.array([[min(max(x, 0), p.nx - 1), 0, min(max(z, 0), p.nz - 1)] for x, z in pts], dtype=np.int32)
    return p


@pytest.mark.parametrize("kind,split", [("elastic2", False), ("elastic2", True), ("em2", False)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,nz,npml,nshots", [(16, 16, 3, 1), (21, 40, 8, 2), (33, 32, 1, 1), (57, 90, 6, 3),
                                               (139, 101, 20, 1), (400, 270, 9, 2)])
def test_regions_equal_one_step_kernel(kind, split, precision, nx, nz, npml, nshots):
    from seidart_amd.solver import Simulation
    p = _ring(tiny_problem(kind, seed=400 + nx, nx=nx, nz=nz, npml=npml, nt=90, nshots=nshots,
                           gamma=1e-3 if kind == "elastic2" else 0.0))
    p.cpml_split = split
    a, b = _walk(p, precision), Simulation(p, precision=precision)
    # segments of every length around the steps per launch, with and without graphs
    for n, gb in ((1, 0), (2, 0), (7, 0), (13, 5), (3, 3), (50, 16), (14, 2)):
        a.run(n)
        b.run(n, graph_block=gb)
        _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
@pytest.mark.parametrize("nx,nz", [(3, 3), (3, 40), (70, 4), (6, 5)])
def test_regions_on_grids_without_slabs(kind, nx, nz):
    """Grids down to 3 x 3 cells without any C-PML slab, the source next to
    and on the outer ring."""
    from seidart_amd.cpml import AxisProfile
    from seidart_amd.solver import Simulation
    base = tiny_problem(kind, seed=420, nx=90, nz=60, npml=2, nt=23, nshots=2)
    p = base
    p.nx, p.nz = nx, nz
    p.coef = {k: v[10:10 + nz, 10:10 + nx].copy() for k, v in p.coef.items()}
    p.prof = {"x": AxisProfile.trivial(nx), "z": AxisProfile.trivial(nz)}
    for q, sh in enumerate(p.shots):
        sh.src = (min(1 + q, nx - 1), 0, min(1, nz - 1)) if q == 0 else (nx - 1, 0, nz - 1)
    _ring(p)
    for precision in ("fp64", "fp32"):
        a, b = _walk(p, precision).run(), Simulation(p, precision=precision).run(graph_block=6)
        _same(a, b)


def test_regions_uneven_models_moments_and_mode_switches():
    from seidart_amd.solver import Simulation
    probs = []
    for m, (nx, nz, npml) in enumerate([(75, 61, 5), (33, 140, 8), (210, 47, 6)]):
        p = _ring(tiny_problem("elastic2", seed=430 + m, nx=nx, nz=nz, npml=npml, nt=64, nshots=2, gamma=1e-3))
        rng = np.random.default_rng(m)
        for sh in p.shots:
            sh.moment = tuple(rng.standard_normal(p.nt) if q in (0, 2, 4) else None for q in range(6))
        probs.append(p)
    a, b = _walk(probs, "fp64"), Simulation(probs, precision="fp64")
    key = (b.steps_per_launch, *b.tiles(), b.tile_order)
    for n, k in ((9, key), (5, (2, 2, 4, 1)), (11, key), (7, (1, 1, 1, 0)), (32, key)):
        b.use(k)
        a.run(n)
        b.run(n, graph_block=4)
        _same(a, b)
    assert float(b.shots[0][2]["trace"].abs().max()) > 0


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
def test_regions_report_the_same_unstable_step(kind):
    from seidart_amd._hip import UnstableError
    from seidart_amd.solver import Simulation
    p = tiny_problem(kind, seed=440, nx=80, nz=70, nt=300)
    p.dt *= 8
    a, b = _walk(p, "fp64").run(), Simulation(p, precision="fp64").run(graph_block=10)
    for s in (a, b):
        with pytest.raises(UnstableError):
            s.check()
    assert a.unstable == b.unstable and a.unstable[0] >= 0


@pytest.mark.parametrize("kind,split", [("elastic2", False), ("elastic2", True), ("em2", False)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,nz,npml,nshots", [(16, 16, 3, 1), (57, 90, 6, 3), (400, 270, 9, 2)])
def test_region_recomputation_equals_one_step_kernel(kind, split, precision, nx, nz, npml, nshots):
    """Every state of a trail (segments of one, of several launches and with a
    remainder) against the one-step kernel stepping the same shots."""
    import ctypes as C

    from seidart_amd import _hip
    from seidart_amd.adjoint import AdjointEngine
    p = _ring(tiny_problem(kind, seed=450 + nx, nx=nx, nz=nz, npml=npml, nt=40, nshots=nshots,
                           gamma=1e-3 if kind == "elastic2" else 0.0))
    p.cpml_split = split
    e = AdjointEngine(p, precision=precision, every=23)
    a = _walk(p, precision)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for it0, n, buf in ((0, 1, 0), (1, 23, 1), (24, 16, 0)):
        for s, (_, _, b) in enumerate(a.shots):
            e.trail[s][buf][0].copy_(b["state"])
        _hip.check(_hip.lib().sdt_plan_run_trail(e.sim._plan, it0, n, buf, st))
        for k in range(1, n + 1):
            a.run(1)
            for s, (_, _, b) in enumerate(a.shots):
                got = e.trail[s][buf][k]
                if kind == "em2":  # Hy's ring, zeroed at the end of a run and read as zero
                    got = got.clone()
                    hy = got[2 * p.cells:3 * p.cells].view(nz, nx)
                    hy[0, : nx - 1] = hy[nz - 2, : nx - 1] = 0
                    hy[: nz - 1, 0] = hy[: nz - 1, nx - 2] = 0
                assert torch.equal(b["state"], got), (it0, k, s)
    a.close()
    e.close()


@pytest.mark.parametrize("nx,nz,npml,nshots", [(400, 270, 9, 3), (803, 611, 13, 1), (660, 23, 6, 18)])
def test_em_regions_of_two_rows_per_thread(nx, nz, npml, nshots):
    """FP32 EM plans of more than 512 regions (two rows per thread, remainders
    of odd heights) against the one-step kernel."""
    from seidart_amd.solver import Simulation
    p = _ring(tiny_problem("em2", seed=460 + nx, nx=nx, nz=nz, npml=npml, nt=48, nshots=nshots))
    a, b = _walk(p, "fp32"), Simulation(p, precision="fp32")
    for n, gb in ((1, 0), (7, 0), (22, 11), (18, 5)):
        a.run(n)
        b.run(n, graph_block=gb)
        _same(a, b)
    a.close()
    b.close()
