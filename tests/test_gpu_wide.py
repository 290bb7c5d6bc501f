"""Kernels by node size: full coupling operators (whole nodes in a wave, one
to four elements a thread, operators all in LDS or bath by bath) and states
above 32 (the product on the matrix cores), and the passes of BiCGSTAB(ell) by
vector length and ell, against the oracle."""

import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import phi_amd as P  # noqa: E402
from oracle import heom_oracle as HO  # noqa: E402

pytestmark = pytest.mark.gpu


def random_state(rng, nodes, N):
    x = rng.normal(size=(nodes, N, N)) + 1j * rng.normal(size=(nodes, N, N))
    return x / np.abs(x).max()


@pytest.mark.parametrize("N,M,terms,lh", [
    (2, 2, 1, 4), (3, 1, 3, 3), (5, 2, 2, 3), (7, 3, 1, 4), (8, 2, 1, 3), (8, 30, 1, 2),
    (9, 2, 1, 3), (16, 1, 2, 3), (17, 2, 1, 2), (22, 2, 1, 2), (23, 1, 1, 3), (24, 1, 2, 2),
    (26, 1, 1, 2)])
def test_full_operators(N, M, terms, lh):
    rng = np.random.default_rng([N, M, terms, lh])
    H = rng.normal(0.0, 0.4, (N, N)) + 0j
    H = H + H.T
    ops = rng.normal(0.0, 0.5, (M, N, N))
    rho0 = np.zeros((N, N), dtype=complex)
    rho0[0, 0] = 1
    kw = dict(gamma=[1.0 + 0.1 * i for i in range(M)], lambda_=[0.05] * M, temperature=0.7,
              lh=lh, num_terms=terms)
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, **kw)
    p.set_int("is_full_bath_coupling", 1)
    p.set_array("bath_coupling_op", np.ascontiguousarray(ops.transpose(0, 2, 1)).reshape(-1))
    assert p.fix("rk4") == 0
    ctx = P.Context(p)
    orc = HO.Oracle(HO.Problem(H=H, rho0=rho0, hbar=1.0, kb=1.0, bath_model="full",
                               bath_ops=ops, **kw))
    x = random_state(rng, ctx.num_nodes, N)
    ref = orc.rhs(x)
    err = np.abs(ctx.rhs(x) - ref).max()
    print("full", N, M, terms, lh, err, np.abs(ref).max(), flush=True)
    # sums of 8 N products a bath and term, each term within the largest sum
    # of magnitudes: 16 N M ulp of it
    big = np.abs(ref).max() * np.sqrt(N) * M
    assert err <= 16 * N * M * 2.2e-16 * big


@pytest.mark.parametrize("N,lh,terms,precision,complex_h", [
    (33, 3, 1, "fp64", True), (34, 2, 2, "fp64", False), (36, 2, 1, "fp64", True),
    (35, 2, 2, "fp32", True)])
def test_more_than_32_states(N, lh, terms, precision, complex_h):
    rng = np.random.default_rng([N, lh, terms])
    H = rng.normal(0.0, 0.4, (N, N)) + 0j
    H = H + H.T
    if complex_h:
        A = rng.normal(0.0, 0.3, (N, N))
        H = H + 1j * (A - A.T)
    M = N  # one site without a bath, one with two
    site = list(range(M))
    site[1] = 0
    rho0 = np.zeros((N, N), dtype=complex)
    rho0[0, 0] = 1
    kw = dict(gamma=[1.0 + 0.02 * i for i in range(M)], lambda_=[0.05] * M, temperature=0.7,
              lh=lh, num_terms=terms)
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    p.set_array("multiple_independent_bath_indices", site)
    p.set_int("is_multiple_independent_baths", 1)
    assert p.fix("rk4") == 0
    ctx = P.Context(p, precision=precision)
    orc = HO.Oracle(HO.Problem(H=H, rho0=rho0, hbar=1.0, kb=1.0, bath_site=site, **kw), threads=4)
    x = random_state(rng, ctx.num_nodes, N)
    x = x + x.conj().transpose(0, 2, 1)   # (the stage kernels' form of Hermitian states)
    x /= np.abs(x).max()
    ctx.set_state(x)
    orc.set_state(x)
    ctx.rk4_steps(3, 0.002)
    orc.rk4(0.006, 0.002, 1.0)
    err = np.abs(ctx.state() - orc.state()).max()
    print("wide", N, lh, terms, precision, err, flush=True)
    # FP32: the increments (|dt L| < 1 of the state) are rounded
    assert err <= (3e-14 if precision == "fp64" else 2e-6)


class Operator:
    """The oracle's steady-state operator as a matrix of krylov_oracle."""

    def __init__(self, orc, shape):
        self.orc, self.shape = orc, shape

    def __matmul__(self, v):
        return self.orc.steady_matvec(v.reshape(self.shape)).reshape(-1)


@pytest.mark.parametrize("N,lh,precision,ell", [
    (2, 2, "fp64", 2),      # fewer elements than a block has threads
    (9, 8, "fp64", 2),      # several trips of the passes
    (36, 2, "fp64", 1), (33, 2, "fp32", 2), (17, 3, "fp64", 3), (5, 4, "fp64", 8)])
def test_steady_state_passes_by_size(N, lh, precision, ell):
    from oracle import krylov_oracle as KO

    rng = np.random.default_rng([N, lh])
    H = rng.normal(0.0, 0.4, (N, N)) + 0j
    H = H + H.T
    rho0 = np.eye(N, dtype=complex) / N
    kw = dict(gamma=[1.0 + 0.02 * i for i in range(N)], lambda_=[0.05] * N, temperature=0.7, lh=lh)
    p = P.params_from_problem(H, rho0, hbar=1.0, kb=1.0, precision=precision, **kw)
    ctx = P.Context(p, precision=precision)
    orc = HO.Oracle(HO.Problem(H=H, rho0=rho0, hbar=1.0, kb=1.0, **kw), threads=4)
    x0 = np.zeros((ctx.num_nodes, N, N), dtype=complex)
    x0[0] = rho0
    b = np.zeros(x0.size, dtype=complex)
    b[0] = 1
    res, _ = KO.bicgstab_l(Operator(orc, x0.shape), b, x0, ell, 2)
    ctx.set_state(x0)
    rc, it, got = ctx.steady_state_l(ell, 1e-30, 2 * ell)
    print("steady", N, lh, precision, ell, got, res[2], flush=True)
    assert it == 2 * ell
    # residuals of the same recurrence, |A|^ell ulp of the first (1e-9 to ell
    # = 2, 1e-8 to 4 where |A| is 20; here |A| < 4)
    assert abs(got - res[2]) <= 1e-8 * res[0]
