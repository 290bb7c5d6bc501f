"""Kernels by node size: full coupling operators (whole nodes in a wave, one
to four elements a thread, operators all in LDS or bath by bath), against
the oracle."""

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
    (9, 2, 1, 3), (16, 1, 2, 3), (17, 2, 1, 2), (22, 2, 1, 2), (23, 1, 1, 3), (24, 1, 2, 2)])
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
