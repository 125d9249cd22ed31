"""Two-pass far field (k_tp_table, k_far_gather) on meshes whose tiles are not the
Kuhn sphere's: tetrahedra in random order, so that a tile of 32 BFs touches up
to 64 distinct tetrahedra (the wide variant), and a last tile of one BF or few."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shuffle", [(1, False), (2, False), (2, True), (3, False), (3, True)])
@pytest.mark.parametrize("omega", [1.3, 1.3 + 0.4j])
def test_far_field_tiles(bfa, orc, torch_cuda, n, shuffle, omega):
    torch = torch_cuda
    V, T = bfa.kuhn_sphere(n, 1.0, 0.05, 77)
    if shuffle:
        T = np.ascontiguousarray(T[np.random.default_rng(1).permutation(len(T))])
    g = bfa.Geometry(V, T)
    g.upload()
    g.build_static(6)
    o = orc.Geometry(V, T)
    M = torch.zeros((g.N, g.N), dtype=torch.complex128, device="cuda")
    g.assemble_vie(omega, bfa.material("iso", eps=4 + 0.1j), M)
    ref = o.assemble(omega, orc.material("iso", eps=4 + 0.1j), g.static_table())
    # the same 64-point sums regrouped: round-off of sums of FP64 products with
    # cancellation (1e-15 measured), far below the desingularised series' 1e-8
    assert np.linalg.norm(M.T.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("omega", [0.3, 3000.0, 2.0e7])
def test_phases_of_any_size(bfa, orc, torch_cuda, omega):
    """The phases' own sine and cosine, small to far beyond any mesh's resolution: rounding of k r is all that is left."""
    torch = torch_cuda
    V, T = bfa.kuhn_sphere(2, 1.0, 0.05, 5)
    g = bfa.Geometry(V, T)
    g.upload()
    g.build_static(6)
    o = orc.Geometry(V, T)
    M = torch.zeros((g.N, g.N), dtype=torch.complex128, device="cuda")
    g.assemble_vie(omega, bfa.material("iso", eps=4 + 0.1j), M)
    ref = o.assemble(omega, orc.material("iso", eps=4 + 0.1j), g.static_table())
    rows, cols = g.touch_pairs()
    far = np.ones((g.N, g.N), bool)
    for a in range(g.N):
        far[a, cols[rows[a]:rows[a + 1]]] = False
    far &= far.T
    d = np.abs(M.T.cpu().numpy() - ref)[far].max() / np.abs(ref[far]).max()
    # both sides round k r to half a unit in the last place, i.e. a phase error
    # of k r 2^-53 each, r <= 2, and the distances differ by a few units (rsqrt)
    assert d <= 1e-12 + 8 * 2 * omega * 2.0 ** -52
