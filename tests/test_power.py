"""Scattered power from tetrahedron currents (bfa_power.hip) against the oracle's
BF-pair sums: every rule (4 points; 16 on a shared vertex; 16 and 33 when k
times a BF's radius exceeds 5), ragged tetrahedron tiles, and the right-hand
side counts at which the kernel's variant changes."""
import numpy as np
import pytest

from conftest import kuhn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,R,omega", [(1, 1.0, 1.0), (2, 1.0, 0.01), (2, 1.0, 1.0), (3, 0.8, 2.5), (3, 1.5, 8.0), (2, 1.5, 40.0)])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 9, 32])
def test_emt_power_against_oracle(bfa, orc, torch_cuda, n, R, omega, nrhs):
    torch = torch_cuda
    V, T = bfa.kuhn_sphere(n, R, 0.05, 21 + n)
    g = bfa.Geometry(V, T)
    g.upload()
    o = orc.Geometry(V, T)
    rng = np.random.default_rng(nrhs)
    spec = []
    for _ in range(nrhs):
        d = rng.standard_normal(3)
        d /= np.linalg.norm(d)
        e = np.cross(d, rng.standard_normal(3))
        spec.append((tuple(e), tuple(d)))
    J = (rng.standard_normal((nrhs, g.N)) + 1j * rng.standard_normal((nrhs, g.N))) * 1e-3
    P = g.emt_power(omega, bfa.planewaves(spec), torch.from_numpy(J).cuda())
    Po = o.emt_power(omega, orc.planewaves(spec), np.ascontiguousarray(J.T))
    # both sum the same products in FP64, about N^2 of them with partial cancellation:
    # N^2 u |largest sum| bounds the difference (N <= 270: 1e-11); rounding is random, 1e-15 measured
    assert np.abs(P - Po).max() <= 1e-12 * np.abs(Po).max()
