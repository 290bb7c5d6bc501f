"""The packed Hermitian stage kernels (RK4 increment form and RKF45 of
Hermitian states) against the full-layout kernels (classic order) and the
oracle: block edges of the packed order, one and two modes per site, real
and complex H, single tiles and long tile sequences, ensembles, and the
changes between the two state layouts."""

import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import phi_amd as P  # noqa: E402
from oracle import heom_oracle as HO  # noqa: E402

pytestmark = pytest.mark.gpu

# One step of either form is the same polynomial; with |dt L| < 1 the FP64
# results differ by a few ulp of the largest entry per step (FP32 bulk: of
# the increments, which are below the state).
TOL = {"fp64": 1e-13, "fp32": 2e-6}


def problem(N, lh, terms, complex_h, seed=0):
    rng = np.random.default_rng([seed, N, lh, terms])
    H = rng.normal(0.0, 0.4, (N, N))
    H = H + H.T + 0j
    if complex_h:
        A = rng.normal(0.0, 0.3, (N, N))
        H = H + 1j * (A - A.T)
    g = rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N))
    rho0 = g @ g.conj().T
    rho0 = (rho0 + rho0.conj().T) / 2
    rho0 /= np.trace(rho0).real
    kw = dict(gamma=[1.0 + 0.1 * i for i in range(N)], lambda_=[0.05] * N, temperature=0.7,
              lh=lh, num_terms=terms)
    return H, rho0, kw


def context(H, rho0, kw, precision):
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    ctx = P.Context(p, precision=precision)
    rng = np.random.default_rng(5)
    x = rng.normal(size=(ctx.num_nodes,) + H.shape) + 1j * rng.normal(
        size=(ctx.num_nodes,) + H.shape)
    x = (x + x.conj().transpose(0, 2, 1)) / 2
    return ctx, x / np.abs(x).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,lh,terms,complex_h", [
    (4, 5, 1, False), (4, 4, 2, True), (5, 4, 1, True), (7, 5, 1, False), (7, 3, 2, False),
    (8, 4, 1, False), (9, 3, 2, True), (13, 3, 1, False), (16, 3, 1, False), (17, 3, 1, True),
    (4, 13, 1, False), (6, 5, 2, True), (7, 9, 1, False), (19, 3, 1, False), (24, 2, 1, False), (24, 3, 1, False)])
def test_packed_steps_equal_the_full_layout(N, lh, terms, complex_h, precision):
    H, rho0, kw = problem(N, lh, terms, complex_h)
    ctx, x = context(H, rho0, kw, precision)
    ctx.set_state(x)
    assert np.array_equal(ctx.state(), x)
    hist = ctx.rk4_history(7, 0.01, 3)
    got = ctx.state()
    ctx.set_rk4_form("classic")
    ctx.set_state(x)
    ref_hist = ctx.rk4_history(7, 0.01, 3)
    ref = ctx.state()
    tol = TOL[precision]
    print(N, lh, terms, precision, np.abs(got - ref).max(), flush=True)
    assert np.abs(got - ref).max() <= tol * 7
    assert np.abs(hist - ref_hist).max() <= tol * 7
    # exactly Hermitian, rho0 read from either layout alike
    assert np.array_equal(got, got.conj().transpose(0, 2, 1))
    assert np.array_equal(ctx.rho0(), ref[0])


@pytest.mark.parametrize("tile,threads,blocks", [(1, 0, 0), (1, 0, 3), (3, 0, 5), (9, 0, 2),
                                                 (10, 256, 3), (16, 256, 1), (20, 0, 7)])
def test_tile_sequences(tile, threads, blocks):
    H, rho0, kw = problem(7, 5, 1, False)
    ctx, x = context(H, rho0, kw, "fp64")
    ctx.set_state(x)
    ctx.rk4_steps(3, 0.01)
    ref = ctx.state()
    ctx.set_launch(2, tile, threads, blocks)
    ctx.set_state(x)
    ctx.rk4_steps(3, 0.01)
    assert np.abs(ctx.state() - ref).max() <= 3e-14


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,terms,depths,blocks", [
    (5, 1, [3, 6, 4, 2, 5], 0), (7, 1, [5, 3, 6, 2], 11), (4, 2, [4, 3, 5], 2),
    (7, 1, [6] * 6 + [3] * 5, 24)])
def test_ensemble_members_equal_single_runs(N, terms, depths, blocks, precision):
    Hs = []
    for m in range(len(depths)):
        H, rho0, kw = problem(N, max(depths), terms, m % 2 == 1, seed=m)
        Hs.append(H)
    p = P.params_from_problem(Hs[0], rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    ens = P.Ensemble(p, Hs, depths, precision=precision)
    if blocks:
        ens.set_launch(2, 2, 0, blocks)   # many tiles and several claims per block
    ens.rk4_steps(70, 0.01)               # eager head, two graph blocks, eager tail
    assert ens.launch_counts()[0] == 64
    got = ens.member_rho0()
    for m, (H, d) in enumerate(zip(Hs, depths)):
        kw["lh"] = d
        q = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
        ctx = P.Context(q, precision=precision)
        x = np.zeros((ctx.num_nodes, N, N), dtype=complex)
        x[0] = rho0
        ctx.set_state(x)
        ctx.rk4_steps(70, 0.01)
        assert np.abs(got[m] - ctx.rho0()).max() <= TOL[precision] * 70


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,terms,members,blocks", [
    (10, 2, 60, 0), (10, 2, 61, 200), (7, 1, 150, 0), (7, 1, 77, 333), (5, 2, 90, 65),
    (6, 1, 5, 0), (7, 1, 3, 5), (4, 1, 2, 0)])
def test_claimed_tiles_equal_one_tile_a_block(N, terms, members, blocks, precision):
    """Every tile is taken once whatever order the blocks' claims come in: the
    results equal, bit for bit, those of a grid of one block per tile."""
    rng = np.random.default_rng([N, members])
    depths = [int(d) for d in rng.integers(2, 5, members)]
    H, rho0, kw = problem(N, max(depths), terms, False)
    Hs = [H + np.diag(rng.normal(0.0, 0.3, N)) for _ in range(members)]
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    out = []
    for grid in (1 << 20, blocks):
        ens = P.Ensemble(p, Hs, depths, precision=precision)
        ens.set_launch(2, 0, 0, grid)
        ens.rk4_steps(70, 0.01)
        out.append(ens.member_rho0())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,tile", [(4, 32), (5, 20), (7, 10), (10, 5)])
def test_graph_blocks_follow_the_launch_shape(N, tile, precision):
    """Graph blocks before and after a change of the shape, also to the tile
    that the full layout takes by default (512 // N^2, the packed one takes
    256 // (N (N + 1) / 2)): the same results as launches one by one."""
    depths = [5, 3, 4, 5, 2, 4, 5, 5]
    Hs = []
    for m in range(len(depths)):
        H, rho0, kw = problem(N, max(depths), 1, False, seed=m)
        Hs.append(H)
    p = P.params_from_problem(Hs[0], rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    out = []
    for graphs in (True, False):
        ens = P.Ensemble(p, Hs, depths, precision=precision)
        ens.set_graphs(graphs)
        runs = []
        for shape in ((), (2, tile), (2, 3), (2, tile), ()):
            ens.set_launch(*shape)
            ens.rk4_steps(70, 0.01)
            assert ens.launch_counts()[0] == (64 if graphs else 0)
            runs.append(ens.state())
        out.append(runs)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,lh", [(5, 5), (16, 3), (17, 3), (20, 2), (24, 2)])
def test_a_single_hierarchy_steps_as_the_only_member(N, lh, precision):
    """One arithmetic for a system, alone or as an ensemble's member, however
    few its nodes are."""
    H, rho0, kw = problem(N, lh, 1, False, seed=2)
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    ens = P.Ensemble(p, [H], [lh], precision=precision)
    ctx = P.Context(p, precision=precision)
    x = np.zeros((ctx.num_nodes, N, N), dtype=complex)
    x[0] = rho0
    ctx.set_state(x)
    ens.rk4_steps(5, 0.01)
    ctx.set_launch(2, 2)                  # the stage kernels for the smallest too
    ctx.rk4_steps(5, 0.01)
    assert np.array_equal(ens.state().reshape(-1), ctx.state().reshape(-1))


def test_states_set_one_after_the_other():
    """Hermitian and other states in turn on one context, each read back as
    set and stepped as on a context of its own."""
    H, rho0, kw = problem(7, 4, 1, False)
    ctx, x = context(H, rho0, kw, "fp64")
    bent = x.copy()
    bent[3, 1, 2] += 0.25j
    for y in (x, bent, bent * 0.5, x * 0.5, x):
        ctx.set_state(y)
        assert np.array_equal(ctx.state(), y)
        assert np.array_equal(ctx.rho0(), y[0])
        ctx.rk4_steps(2, 0.01)
        one, _ = context(H, rho0, kw, "fp64")
        one.set_state(y)
        one.rk4_steps(2, 0.01)
        assert np.array_equal(ctx.state(), one.state())
        ctx.set_state(x * 2.0)            # and one that is never stepped


def test_a_state_that_is_not_hermitian_takes_the_full_layout():
    H, rho0, kw = problem(7, 4, 1, False)
    ctx, x = context(H, rho0, kw, "fp64")
    x[3, 1, 2] += 0.25j
    ctx.set_state(x)
    ctx.rk4_steps(5, 0.01)
    got = ctx.state()
    ctx.set_launch(1, 0, 0, 0)            # one-shot kernels: nested order, full layout
    ctx.set_state(x)
    ctx.rk4_steps(5, 0.01)
    assert np.abs(got - ctx.state()).max() <= 1e-13
    # and a Hermitian state set afterwards is stepped as one again
    ctx.set_launch()
    y = (x + x.conj().transpose(0, 2, 1)) / 2
    ctx.set_state(y)
    ctx.rk4_steps(5, 0.01)
    assert np.array_equal(ctx.state(), ctx.state().conj().transpose(0, 2, 1))


def test_tuned_shapes_are_kept_per_layout():
    """A shape tuned on a state that is not Hermitian (full layout) is not the
    answer for a Hermitian one of the same sizes; another Hermitian context
    gets the kept one."""
    H, rho0, kw = problem(6, 6, 1, False)
    ms = []
    for bend in (0.25j, 0, 0):
        ctx, x = context(H, rho0, kw, "fp64")
        x[2, 0, 1] += bend
        ctx.set_state(x)
        ms.append(ctx.autotune(0.001, steps=2)[0])
        assert np.array_equal(ctx.state(), x)
    assert ms[0] != ms[1] == ms[2]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_layout_changes_between_calls(precision):
    """RK4, an RKF45 attempt, an accepted one, the RHS and the autotuner on one
    context, against the oracle's stepping of the same sequence."""
    H, rho0, kw = problem(6, 4, 1, False)
    ctx, _ = context(H, rho0, kw, precision)
    x = np.zeros((ctx.num_nodes, 6, 6), dtype=complex)
    x[0] = rho0
    dt = 0.01
    b = np.array([2. / 9., 1. / 12., 1. / 4., 69. / 128., -243. / 128., 135. / 64., -17. / 12.,
                  27. / 4., -27. / 5., 16. / 15., 65. / 432., -5. / 16., 13. / 16., 4. / 27.,
                  5. / 144., 1. / 9., 9. / 20., 16. / 45., 1. / 12., 47. / 450., 12. / 25.,
                  32. / 225., 1. / 30., 6. / 25.]) * dt
    ctx.set_state(x)
    ctx.rk4_steps(2, dt)
    ctx.rkf45_attempt(b)              # not accepted: the state stays
    before = ctx.state()
    ctx.rk4_steps(1, dt)
    ctx.rkf45_attempt(b)
    ctx.rkf45_accept()
    ctx.autotune(dt, steps=1)
    nodes = ctx.rhs_nodes([0, 3])
    got = ctx.state()
    orc = HO.Oracle(HO.Problem(H, rho0, hbar=1.0, kb=1.0, **kw))
    orc.rk4(2 * dt - dt / 2, dt, 1.0)
    tol = 1e-12 if precision == "fp64" else 1e-6
    assert np.abs(before - orc.state()).max() <= tol
    assert np.abs(nodes - orc.rhs(got)[[0, 3]]).max() <= 1e-12

    def rk4(y):
        k0 = orc.rhs(y)
        k1 = orc.rhs(y + dt / 2 * k0)
        k2 = orc.rhs(y + dt / 2 * k1)
        k3 = orc.rhs(y + dt * k2)
        return y + dt / 6 * (k0 + 2 * k1 + 2 * k2 + k3)

    # RK4 and the 5th-order Fehlberg step agree to dt^5 |L|^5 / 120
    assert np.abs(got - rk4(rk4(orc.state()))).max() <= 1e-9 + tol


@pytest.mark.parametrize("N,tile", [(4, 64), (5, 40), (7, 20)])
def test_packed_steps_after_an_accepted_full_layout_attempt(N, tile):
    """An accepted RKF45 attempt on the full layout exchanges the state with
    the buffer that packed stages use next: tiles larger than the slab."""
    H, rho0, kw = problem(N, 2, 1, False)
    ctx, x = context(H, rho0, kw, "fp64")
    ctx.set_launch(2, tile)
    ctx.set_state(x)
    ctx.rk4_steps(3, 0.01)
    ref = ctx.state()
    bent = x.copy()
    bent[1, 0, 1] += 0.5j                 # not Hermitian
    ctx.set_state(bent)
    ctx.rkf45_attempt(np.full(24, 0.001))
    ctx.rkf45_accept()
    ctx.set_state(x)
    ctx.rk4_steps(3, 0.01)
    assert np.array_equal(ctx.state(), ref)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,lh,terms,complex_h", [
    (1, 9, 1, False), (2, 9, 2, False), (2, 2, 1, True), (3, 4, 2, True), (3, 8, 1, False),
    (4, 6, 1, True), (5, 3, 2, False), (7, 3, 1, False), (8, 2, 1, True)])
def test_one_workgroup_steps_equal_the_stage_kernels(N, lh, terms, complex_h, precision):
    H, rho0, kw = problem(N, lh, terms, complex_h, seed=3)
    ctx, x = context(H, rho0, kw, precision)
    ctx.set_state(x)
    hist = ctx.rk4_history(23, 0.01, 4)
    ctx.rk4_steps(1, 0.01)
    got = ctx.state()
    ctx.set_rk4_form("classic")           # the full-layout stage kernels
    ctx.set_state(x)
    ref_hist = ctx.rk4_history(23, 0.01, 4)
    ctx.rk4_steps(1, 0.01)
    tol = TOL[precision] * 24
    assert hist.shape == ref_hist.shape == (6, N, N)
    assert np.abs(hist - ref_hist).max() <= tol
    assert np.abs(got - ctx.state()).max() <= tol
    assert np.array_equal(got, got.conj().transpose(0, 2, 1))


def test_one_workgroup_runs_longer_than_a_launch_match_the_oracle():
    """5000 steps (two launches) and the autotuner, which leaves the state."""
    H, rho0, kw = problem(2, 4, 1, False, seed=4)
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, **kw)
    ctx = P.Context(p)
    x = np.zeros((ctx.num_nodes, 2, 2), dtype=complex)
    x[0] = rho0
    ctx.set_state(x)
    ms, shape = ctx.autotune(0.001, steps=5)
    assert ms > 0 and np.array_equal(ctx.state(), x)
    # the shape it gives sets the same kernel: no graph blocks of stage kernels
    other = P.Context(p)
    other.set_launch(*shape)
    other.set_state(x)
    other.rk4_steps(70, 0.001)
    assert other.launch_counts() == (0, 70)
    hist = ctx.rk4_history(5000, 0.001, 500)
    assert hist.shape[0] == 10
    orc = HO.Oracle(HO.Problem(H, rho0, hbar=1.0, kb=1.0, **kw))
    orc.rk4(5.0 - 0.0005, 0.001, 10.0)
    assert np.abs(ctx.state() - orc.state()).max() <= 1e-10
