"""The diagnostics' per-element sums bit for bit: entropy is a difference of logarithms
that cancels on isentropic flow, so its digits are those of the logarithm, and no other
formula for it may take the place of log((gamma - 1) rho e) - gamma log(rho) with the
math library's logarithm (torch's, on the same device) and IEEE division.

One node of each element is rough, the others are at rho = 1, rho e = 1 / (gamma - 1),
whose entropy and kinetic energy are exact zeros; the element's sums are then its rough
node's terms, whose few rounded operations are repeated here.  About one logarithm in 50 of
another formula differs in its last bit: 640 elements or more per shape."""

from fractions import Fraction

import numpy as np
import pytest
import torch

from helpers import small_problem

pytestmark = pytest.mark.gpu

GAMMA = 1.5        # gamma - 1 and 1 / (gamma - 1) are exact


def fma(a, b, c):
    """a b + c with one rounding."""
    return float(Fraction(a) * Fraction(b) + Fraction(c))


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 3), (2, 5), (3, 2), (3, 3), (3, 4)])
def test_per_element_sums_are_those_of_the_library_functions(dim, N):
    prob = small_problem(dim, N)
    print(f"case diagnostics bits dim={dim} N={N} K={prob.K}", flush=True)
    rng = np.random.default_rng(dim * 10 + N)
    for _ in range(-(-640 // prob.K)):
        check(prob, rng)


def check(prob, rng):
    from scratch_wadge_amd import _lib
    dim, N, K, Nq = prob.dim, prob.N, prob.K, prob.Nq
    rho = rng.uniform(0.2, 3.0, K)
    m = rng.standard_normal((dim, K))
    E = rng.uniform(4.0, 30.0, K) / rho + 0.5 * (m * m).sum(0) / rho
    node = rng.integers(0, Nq, K)
    Q = np.zeros((K, dim + 2, Nq))
    Q[:, 0], Q[:, -1] = 1.0, 1.0 / (GAMMA - 1.0)
    k = np.arange(K)
    Q[k, 0, node], Q[k, -1, node] = rho, E
    for d in range(dim):
        Q[k, 1 + d, node] = m[d]

    mm = m[0] * m[0]
    for d in range(1, dim):
        mm = np.array([fma(x, x, y) for x, y in zip(m[d], mm)])
    rhoe = E - 0.5 * mm / rho
    log = lambda x: torch.log(torch.as_tensor(x, device="cuda")).cpu().numpy()
    s = np.array([fma(-GAMMA, lr, lp) for lr, lp in zip(log(rho), log((GAMMA - 1.0) * rhoe))])
    wJ = prob.wq[node] * prob.Jq.reshape(K, Nq)[k, node]
    kinetic, entropy = 0.5 * mm / rho * wJ, wJ * (-rho * s)

    D = lambda a: torch.as_tensor(np.ascontiguousarray(a).reshape(-1), dtype=torch.float64, device="cuda")
    wq, Jq, Qd, aux, tot = D(prob.wq), D(prob.Jq), D(Q), D(np.zeros(4 * K)), D(np.zeros(4))
    plan = _lib.Plan(dim, N, Nq, prob.Nfq, GAMMA, 1.0)
    plan.diagnostics(K, *(t.data_ptr() for t in (wq, Jq, Qd)), None, aux.data_ptr(), tot.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    got = aux.cpu().numpy().reshape(K, 4)
    assert np.array_equal(got[:, 0], kinetic)
    assert np.array_equal(got[:, 1], entropy)
    assert np.all(got[:, 2] == 0.0)
