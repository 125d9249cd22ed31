"""Fields from tetrahedron currents: points where the basis functions of one
tetrahedron are on different rules, and both sizes of a workgroup's chunk,
against the oracle's sum over basis functions."""
import numpy as np
import pytest

from conftest import kuhn
from test_fields import _fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,npts", [(1, 1), (3, 7), (1, 1100)])
def test_mixed_rules_match_oracle(bfa, orc, torch_cuda, n, npts):
    V, T = kuhn(bfa, n)
    g = bfa.Geometry(V, T)
    g.upload()
    o = orc.Geometry(V, T)
    rng = np.random.default_rng(100 * n + npts)
    J = rng.standard_normal(g.N) + 1j * rng.standard_normal(g.N)
    d = rng.standard_normal((npts, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    # the rules change where the distance is ten radii of a basis function
    X = V.mean(axis=0) + d * np.exp(rng.uniform(np.log(1.5), np.log(30.0), npts))[:, None]
    E, H = _fields(bfa, torch_cuda, g, 1.7, X, J)
    ref = orc.fields(o, V, T, J, 1.7, X, [])
    for got, want in ((E, ref[:, :3]), (H, ref[:, 3:])):
        scale = np.abs(want).max(axis=1)
        # N terms of random sign, each good to a few eps
        assert (np.abs(got - want).max(axis=1) / scale).max() < 1e-12
