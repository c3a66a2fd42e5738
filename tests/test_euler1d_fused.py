"""The fused 1D RK2 step (m3p_euler1d_rk2_step_blocks, one launch per step,
the first stage's state never stored) against the two work-list stage
launches it replaces: the same arithmetic on the same operands, so every
value must be equal (==), for every block size, on the full 512-problem
ensemble, on a ring (periodic) chain and at outflow ends.  The _cfl form
leaves the time step the separate reduction computes from its output, bit
for bit, and its hipGraph replays equal eager two-stage steps with separate
reductions.  Tables whose prev/next links are not mutual are refused."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")]


def _pair(count, n, lmin, lmax, seed=3):
    from mara3p_amd import problems
    from mara3p_amd.solvers import Euler1DEnsembleSolver
    mesh, u0 = problems.riemann_ensemble(count=count, block_size=n, lmin=lmin, lmax=lmax, seed=seed)
    a = Euler1DEnsembleSolver(mesh, gamma=1.4, plm_theta=1.5, precision="mixed")
    b = Euler1DEnsembleSolver(mesh, gamma=1.4, plm_theta=1.5, precision="mixed")
    a.set_state(u0)
    b.set_state(u0)
    return a, b


def _steps_equal(a, b, steps):
    dt = float(a.cfl_dt(0.4).item())
    for _ in range(steps):
        a.step(dt)
        b.step_fused(dt)
    a.check_errors()
    b.check_errors()
    ua, ub = a.state(), b.state()
    assert np.array_equal(ua, ub), float(np.abs(ua - ub).max())


@pytest.mark.parametrize("n", [16, 32, 64, 128, 256, 512])
def test_fused_rk2_equals_two_stages(n):
    """Three RK2 steps, fused against two stage launches each, on an
    ensemble of 12 problems of 2 to 16 blocks (outflow ends, one cell
    spacing per problem): equal in every value.  n = 512 runs two tiles of
    256 zones per block."""
    a, b = _pair(12, n, 2 * n, 16 * n, seed=5 + n)
    _steps_equal(a, b, 3)


def test_fused_rk2_equals_two_stages_full_ensemble():
    """The 512-problem ensemble of 512 to 8192 zones in blocks of 64: two
    steps, equal in every value."""
    a, b = _pair(512, 64, 512, 8192, seed=1)
    _steps_equal(a, b, 2)


def test_fused_rk2_ring():
    """One problem of 6 blocks closed into a ring (periodic ends, the links
    rewritten on both solvers): equal in every value after three steps."""
    a, b = _pair(1, 64, 384, 384, seed=9)
    for s in (a, b):
        nbr = s.nbr.clone()
        nbr[0, 0] = s.mesh.nblk - 1
        nbr[s.mesh.nblk - 1, 1] = 0
        s.nbr = nbr
    _steps_equal(a, b, 3)


def test_fused_rk2_cfl_output_and_dt():
    """The _cfl form: the output of the plain fused step, and dt_next equal
    to the separate reduction of that output (m3p_euler_cfl_dt_blocks)."""
    a, _ = _pair(16, 64, 128, 1024, seed=7)
    dt = a.cfl_dt(0.4)
    out_plain = torch.empty_like(a.u)
    out_cfl = torch.empty_like(a.u)
    dt_next = torch.zeros(1, dtype=torch.float64, device="cuda")
    a.rk2_step(a.u, out_plain, 0.0, dt_dev=dt)
    a.rk2_step(a.u, out_cfl, 0.0, dt_dev=dt, cfl=0.4, dt_next=dt_next)
    a.check_errors()
    assert torch.equal(out_plain, out_cfl)
    a.u = out_cfl
    sep = float(a.cfl_dt(0.4).item())
    assert float(dt_next.item()) == sep
    assert 0.0 < sep < 1.0


def test_fused_rk2_cfl_graph_replays_match_eager_separate():
    """A hipGraph of two fused CFL steps replayed three times with eager work
    between the replays, against the same steps issued eagerly as two stage
    launches with a separate CFL reduction before each step: the state and
    the time step after every replay, bit for bit."""
    from mara3p_amd.solvers import Graph, cfl_step_pair, cfl_step_pair_rk2
    g_s, e_s = _pair(16, 64, 128, 1024, seed=11)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        g_s.cfl_dt(0.4)
        with Graph() as g:
            cfl_step_pair_rk2(g_s, 0.4)
    stream.synchronize()
    torch.cuda.synchronize()
    for rep in range(3):
        with torch.cuda.stream(stream):
            g.replay()
        stream.synchronize()
        cfl_step_pair(e_s, 0.4)
        torch.cuda.synchronize()
        _ = torch.ones(1024, device="cuda").sum().item()      # eager work between replays
        assert np.array_equal(g_s.state(), e_s.state()), rep
        assert float(g_s.dt_dev.item()) == float(e_s.cfl_dt(0.4).item()), rep
    g_s.check_errors()
    e_s.check_errors()
    del g


@pytest.mark.parametrize("n", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("order", ["storage", "reversed", "shuffled"])
def test_fused_rk2_windows_follow_the_links(n, order):
    """Windows of 56 zones over tables whose links leave the storage order:
    chains of two to nine blocks (shorter and longer than a window), rings of
    one and three blocks, their blocks stored in order, backwards and shuffled,
    each with its own cell spacing.  Equal in every value to two stage
    launches, and the CFL form to the separate reduction."""
    from mara3p_amd.mesh import EnsembleMesh1D
    from mara3p_amd.solvers import Euler1DEnsembleSolver
    rng = np.random.default_rng(n)
    chains, rings = [2, 9, 3, 2, 5], [1, 3]
    total = sum(chains) + sum(rings)
    where = {"storage": np.arange(total), "reversed": np.arange(total)[::-1], "shuffled": rng.permutation(total)}[order]
    nbr, dl, first = np.full((total, 2), -1, np.int32), np.empty(total), 0
    for m, ring in [(m, False) for m in chains] + [(m, True) for m in rings]:
        for k in range(m):
            b = where[first + k]
            if k > 0 or ring:
                nbr[b, 0] = where[first + (k - 1) % m]
            if k < m - 1 or ring:
                nbr[b, 1] = where[first + (k + 1) % m]
            dl[b] = 1.0 / (m * n)
        first += m
    s = Euler1DEnsembleSolver(EnsembleMesh1D([total * n], n), precision="mixed")
    s.nbr.copy_(torch.as_tensor(nbr))
    s.dl.copy_(torch.as_tensor(dl))
    rho, v, p = 1.0 + rng.random((total, n)), 0.5 * rng.standard_normal((total, n)), 0.5 + rng.random((total, n))
    u0 = np.stack([rho, rho * v, 0 * v, 0.1 * rho, 0.5 * rho * (v * v + 0.01) + p / 0.4], axis=1)
    s.set_state(u0)
    dt = 0.02 / (9 * n)
    s.stage(s.u, None, s.u1, dt)
    s.stage(s.u1, s.u, s.u2, dt)
    out = torch.empty_like(s.u)
    dt_next = torch.zeros(1, dtype=torch.float64, device="cuda")
    s.rk2_step(s.u, out, dt)
    assert torch.equal(out, s.u2)
    out.zero_()
    s.rk2_step(s.u, out, dt, cfl=0.4, dt_next=dt_next)
    s.check_errors()
    assert torch.equal(out, s.u2)
    s.u = out
    assert float(dt_next.item()) == float(s.cfl_dt(0.4).item())


def test_fused_rk2_refuses_what_it_does_not_compute():
    """FP64, a block size outside the list and aliasing are refused before
    any launch; a one-block problem (prev outflow, next itself: links that
    are not mutual) is refused by the solver on the host and, through the C
    ABI, reported by the kernel as M3P_ERR_BAD_SHAPE."""
    from mara3p_amd import problems
    from mara3p_amd._lib import M3PError, lib
    from mara3p_amd.mesh import EnsembleMesh1D
    from mara3p_amd.solvers import Euler1DEnsembleSolver
    L = lib()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def call(s, u, out, n):
        return L.m3p_euler1d_rk2_step_blocks(ctypes.c_void_p(u.data_ptr()), ctypes.c_void_p(out.data_ptr()),
                                             ctypes.c_void_p(s.nbr.data_ptr()), ctypes.c_void_p(s.dl.data_ptr()),
                                             s.mesh.nblk, n, 1e-4, ctypes.c_void_p(0), 0.5, s.theta, s.gamma,
                                             s.precision, stream)
    mesh, u0 = problems.riemann_ensemble(count=4, block_size=64, lmin=128, lmax=256, seed=2)
    s64 = Euler1DEnsembleSolver(mesh, precision="fp64")
    assert call(s64, s64.u, s64.u2, 64) != 0
    sm = Euler1DEnsembleSolver(mesh, precision="mixed")
    assert call(sm, sm.u, sm.u2, 48) != 0
    assert call(sm, sm.u, sm.u, 64) != 0
    # one problem of one block, one of three
    one = Euler1DEnsembleSolver(EnsembleMesh1D([64, 192], 64), precision="mixed")
    assert not one.links_mutual()
    with pytest.raises(ValueError):
        one.step_fused(1e-4)
    one.u.copy_(torch.as_tensor(np.concatenate([u0[:1], u0[:3]]), device="cuda"))
    assert call(one, one.u, one.u2, 64) == 0
    with pytest.raises(M3PError) as e:
        one.check_errors()
    assert e.value.code == 4


@pytest.mark.parametrize("n", [16, 64, 256])
def test_fused_rk2_neighbours_behind_the_list(n):
    """A list whose outer neighbours are stored behind it (with rows of their own
    in the link table and the cell spacings): its blocks equal the same blocks
    of the whole chain's fused step, and a negative density in any of the four
    guard zones there is reported."""
    from mara3p_amd._lib import M3P_MIXED, NegativeDensityError, check, check_kernel_errors, lib
    rng = np.random.default_rng(n)
    m = 7
    rho, v, p = 1 + rng.random((m, n)), 0.5 * rng.standard_normal((m, n)), 0.5 + rng.random((m, n))
    u = np.stack([rho, rho * v, 0 * v, 0.1 * rho, 0.5 * rho * (v * v + 0.01) + p / 0.4], axis=1)
    dl = (1.0 + rng.random(m)) / (m * n)
    dt = 0.05 * dl.min()
    dev = lambda x, t: torch.as_tensor(np.ascontiguousarray(x), dtype=t, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def step(state, nbr, spacing, k):
        us, ns, ds = dev(state, torch.float64), dev(nbr, torch.int32), dev(spacing, torch.float64)
        out = torch.empty((k, 5, n), dtype=torch.float64, device="cuda")
        check(lib().m3p_euler1d_rk2_step_blocks(us.data_ptr(), out.data_ptr(), ns.data_ptr(), ds.data_ptr(), k, n,
                                                dt, None, 0.5, 1.5, 1.4, M3P_MIXED, stream))
        check_kernel_errors(stream)
        return out.cpu().numpy()

    b = np.arange(m)
    chain = np.stack([b - 1, np.where(b < m - 1, b + 1, -1)], axis=1)
    whole = step(u, chain, dl, m)
    # blocks 1 .. m - 2 of the chain as a list, block 0 and block m - 1 behind it
    order = np.concatenate([b[1:-1], [0, m - 1]])
    at = np.argsort(order)
    table = np.where(chain[order] >= 0, at[np.maximum(chain[order], 0)], -1)
    assert np.array_equal(step(u[order], table, dl[order], m - 2), whole[1:-1])
    for block, zone in ((m - 2, n - 4), (m - 2, n - 1), (m - 1, 0), (m - 1, 3)):
        bad = u[order].copy()
        bad[block, 0, zone] = -1.0
        with pytest.raises(NegativeDensityError):
            step(bad, table, dl[order], m - 2)
