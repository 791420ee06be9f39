"""Which kernels a run takes (sdt_plan_get_run_mode: 0 one step per launch, 1
two, 2 regions), and that each of them is the one that a caller asked for."""
import numpy as np
import pytest
import torch

from helpers import tiny_problem

pytestmark = pytest.mark.gpu


def _problem(kind, seed, nt, **kw):
    p = tiny_problem(kind, seed=seed, nt=nt, nrec=9, **kw)
    for sh in p.shots:  # the corners and the source cell too
        i, _, k = sh.src
        sh.rec = np.concatenate([sh.rec, np.array([[0, 0, 0], [p.nx - 1, 0, p.nz - 1], [i, 0, k]], dtype=np.int32)])
    return p


def _same(a, b):
    torch.cuda.synchronize()
    for (_, _, x), (_, _, y) in zip(a.shots, b.shots):
        assert torch.equal(x["state"], y["state"])
        assert torch.equal(x["trace"], y["trace"])


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
def test_a_launch_shape_that_is_set_runs(kind):
    """Also one that the plan had already: every setter leaves the regions."""
    from seidart_amd.solver import Simulation
    s = Simulation(_problem(kind, 500, 60, nx=70, nz=50, npml=5), precision="fp32")
    own = (s.steps_per_launch, *s.tiles(), s.tile_order)
    assert s.regions and s.run_mode(60) == 2 and s.run_mode(60, 20) == 2
    for set_own in (lambda: setattr(s, "steps_per_launch", own[0]), lambda: s.set_tiles(*own[1:3]),
                    lambda: setattr(s, "tile_order", own[3])):
        set_own()
        assert not s.regions and s.run_mode(60) == own[0] - 1
        s.use(own)
        assert s.regions and s.run_mode(60) == 2
    s.steps_per_launch = 1
    assert s.run_mode(60) == 0
    s.steps_per_launch = 2
    assert (s.run_mode(60), s.run_mode(60, 20), s.run_mode(60, 15), s.run_mode(1)) == (1, 1, 0, 0)
    s.regions = True
    assert s.run_mode(60) == 2
    s.regions = False
    assert s.run_mode(60) == 1
    s.close()


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("tiles", [None, (1, 2), (4, 8)])
def test_two_step_kernel_over_segments(kind, precision, tiles):
    """The two-step kernel over odd segments, odd and even graph blocks, from
    odd steps and after switches, against the one-step kernel."""
    from seidart_amd.solver import Simulation
    p = _problem(kind, 510, 64, nx=150, nz=75, npml=6, nshots=2)
    a, b = Simulation(p, precision=precision), Simulation(p, precision=precision)
    a.use((1, 4, 32, 0))
    b.steps_per_launch = 2
    if tiles:
        b.set_tiles(*tiles)
    for n, gb, mode in ((1, 0, 0), (3, 0, 1), (6, 4, 1), (5, 5, 0), (9, 2, 1), (2, 2, 1), (11, 11, 0), (8, 8, 1)):
        assert b.run_mode(n, gb) == mode and a.run_mode(n, gb) == 0
        a.run(n)
        b.run(n, graph_block=gb)
        _same(a, b)
    b.regions = True   # regions and back
    a.run(7)
    b.run(7)
    b.regions = False
    a.run(12)
    b.run(12, graph_block=4)
    _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_short_runs_take_the_walking_kernels(kind, precision):
    """A run or graph block of too few steps for a region's halo goes to the
    walkers (one step: every plan), longer ones to regions, with the same bits
    whatever the sequence."""
    from seidart_amd.solver import Simulation
    p = _problem(kind, 520, 46, nx=90, nz=60, npml=6)
    a, b = Simulation(p, precision=precision), Simulation(p, precision=precision)
    a.use((1, 4, 32, 0))
    assert [b.run_mode(n) for n in (1, 2, 3, 50)] == [0, 2, 2, 2]
    assert b.run_mode(10, 2) != 2 and b.run_mode(12, 3) == b.run_mode(50, 50) == 2
    for n, gb in ((1, 0), (1, 0), (2, 0), (1, 0), (4, 2), (5, 0), (1, 0), (1, 1), (9, 3), (1, 0), (6, 2), (13, 13), (1, 0)):
        a.run(n)
        b.run(n, graph_block=gb)
        _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_short_runs_of_many_regions(kind, precision):
    """More than 4096 regions: pairs of steps on the two-step kernel, the plan
    path and the allocation-free one."""
    from seidart_amd.solver import Simulation
    p = _problem(kind, 530, 30, nx=400, nz=300, npml=6, nshots=34)
    p.cpml_split = kind == "elastic2"
    a, b, c = (Simulation(p, precision=precision) for _ in range(3))
    assert b.region_info()[2] > 4096
    a.use((1, 4, 32, 0))
    assert [b.run_mode(n) for n in (1, 2, 5, 50)] == [0, 1, 2, 2]
    assert b.run_mode(4, 4) == 1 and b.run_mode(50, 10) == 2
    for n, gb in ((2, 0), (1, 0), (2, 0), (4, 4), (5, 0), (2, 0), (1, 0), (8, 2), (5, 0)):
        a.run(n)
        b.run(n, graph_block=gb)
        c.run_noalloc(n)
        _same(a, b)
        _same(a, c)
    for s in (a, b, c):
        s.close()


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,nz,offset", [(33, 21, 0), (33, 21, 1), (40, 28, 3), (130, 97, 2)])
def test_copies_between_the_state_buffers(kind, precision, nx, nz, offset):
    """Runs that end in buffer B are copied back, and the copy a one-step run
    from an odd step needs in B is made, also for arrays off the 16-byte grid
    and for buffers that are aligned differently (B shifted by `offset`
    elements)."""
    from seidart_amd.solver import Simulation
    p = _problem(kind, 540 + nx, 16, nx=nx, nz=nz, npml=4, nshots=2)
    a, b = Simulation(p, precision=precision), Simulation(p, precision=precision)
    a.use((1, 4, 32, 0))
    keep, el = [], b.shots[0][2]["state"].element_size()
    for S, (_, _, bufs) in zip(b._shots, b.shots):
        n = bufs["state"].numel()
        st = torch.full((n + offset + 8,), 7.0, dtype=b.dtype, device=b.device)
        st[offset:offset + n] = bufs["state"]
        keep.append(st)
        for f in range(len(b.names)):
            S.field_b[f] = st.data_ptr() + (offset + f * p.nx * p.nz) * el
        S.psi_b = st.data_ptr() + (offset + len(b.names) * p.nx * p.nz) * el
    for n in (1, 1, 3, 1, 2, 1, 5, 1):  # (the last two from odd steps)
        a.run(n)
        b.run_noalloc(n)
        _same(a, b)
    for st in keep:  # nothing written past B
        assert float(st[-8:].min()) == float(st[-8:].max()) == 7.0
        assert offset == 0 or float(st[:offset].min()) == 7.0
    a.close()
    b.close()


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_profile_times_the_kernels_that_run_takes(kind, precision):
    """In each mode: the state that a run of as many steps leaves, and the time
    of the kernel per launch in the first slot."""
    from seidart_amd.solver import Simulation
    p = _problem(kind, 560, 120, nx=300, nz=260, npml=6, nshots=2)
    a, b = Simulation(p, precision=precision), Simulation(p, precision=precision)
    a.use((1, 4, 32, 0))
    most = b.region_info()[1]
    for setup, n in ((None, 3 * most), (None, 2 * most - 1), (2, 6), (2, 7), (1, 5), (None, 1)):
        if setup:
            b.steps_per_launch = setup
        else:
            b.regions = True
        mode = b.run_mode(n)
        assert mode == (0 if n == 1 else 2 if setup is None else setup - 1)
        a.run(n)
        ms = b.profile(n)
        _same(a, b)
        assert ms[0] > 0 and ms[1] >= 0 and ms[2] >= 0
        if mode:
            assert ms[1] == ms[2] == 0
    a.close()
    b.close()


@pytest.mark.parametrize("nx,nz,nshots", [(660, 23, 20), (23, 691, 20), (47, 31, 140)])
def test_em_regions_of_two_rows_on_thin_grids(nx, nz, nshots):
    """FP32 EM plans of more than 512 regions (two rows per thread) whose
    regions overhang a thin grid on both sides, its height odd, against the
    one-step kernel."""
    from seidart_amd.solver import Simulation
    p = _problem("em2", 570 + nx, 40, nx=nx, nz=nz, npml=6, nshots=nshots)
    a, b = Simulation(p, precision="fp32"), Simulation(p, precision="fp32")
    on, most, count = b.region_info()
    assert on and count > 512 and 3 <= most <= 8
    a.use((1, 4, 32, 0))
    for n, gb in ((7, 0), (22, 11), (11, 5)):
        assert b.run_mode(n, gb) == 2
        a.run(n)
        b.run(n, graph_block=gb)
        _same(a, b)
    a.close()
    b.close()


def _copies(kind, seed, nt, n):
    """n equal shots on one model: more items than one launch takes (262,144)."""
    p = _problem(kind, seed, nt, nx=600, nz=500, npml=6)
    return p, p.with_shots(list(p.shots) * n)


@pytest.mark.parametrize("kind", ["elastic2", "em2"])
def test_regions_in_several_launches(kind):
    """A list of more regions than one launch takes: every shot equals the
    shot alone, bit for bit."""
    from seidart_amd.solver import Simulation
    one, many = _copies(kind, 580, 12, 510)
    a, b = Simulation(one, precision="fp32"), Simulation(many, precision="fp32")
    assert b.region_info()[2] > 1 << 18 and b.run_mode(12, 10) == 2
    a.run()
    b.run(graph_block=10).check()
    torch.cuda.synchronize()
    ref = a.shots[0][2]
    assert float(ref["trace"].abs().max()) > 0
    for _, _, x in b.shots:
        assert torch.equal(x["state"], ref["state"]) and torch.equal(x["trace"], ref["trace"])
    a.close()
    b.close()


def test_recomputation_and_adjoint_in_several_launches():
    """The same of the trail recomputation and the adjoint: lambda_0 of every
    shot equals that of the shot alone, and the gradient is their sum."""
    from seidart_amd.adjoint import AdjointEngine
    one, many = _copies("em2", 590, 10, 520)
    lam, grad = [], []
    for p in (one, many):
        e = AdjointEngine(p, precision="fp32", every=5)
        tr = e.forward()
        g, _ = e.backward([t + 1.0 for t in tr])
        grad.append(g[0].cpu())
        lam.append([e.adjoint_state(s) for s in range(len(p.shots))])
        keep = lam[0][0].clone()
        if p is many:
            for s, x in enumerate(lam[1]):
                assert torch.equal(x, ref), s
        ref = keep
        e.close()
    assert float(ref.abs().max()) > 0
    n, scale = len(many.shots), grad[0].abs().amax(dim=(1, 2), keepdim=True)
    # FP32 atomics: n values of one size per step and cell, 10 steps, in any order
    assert float(((grad[1] - n * grad[0]).abs() / (n * scale)).max()) < 10 * n * 2.0 ** -24
