"""Assemblies of one geometry with different materials on two streams: the
geometry's Gram blocks serve them in turn."""
import numpy as np
import pytest

from conftest import kuhn

pytestmark = pytest.mark.gpu


def test_two_streams_two_materials(bfa, torch_cuda):
    torch = torch_cuda
    V, T = kuhn(bfa, 4)
    g = bfa.Geometry(V, T)
    g.upload()
    g.build_static(6)
    mats = [bfa.material("diag", eps=(4 + 0.05j, 5 + 0.05j, 6 + 0.05j)), bfa.material("iso", eps=9 + 1j)]
    new = lambda: torch.zeros((g.N, g.N), dtype=torch.complex128, device="cuda:0")
    ref = [new(), new()]
    for m, r in zip(mats, ref):
        g.assemble_vie(1.0, m, r)
        torch.cuda.synchronize()
    assert (ref[0] - ref[1]).abs().max() > 0
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    out = [[new() for _ in range(6)] for _ in mats]
    torch.cuda.synchronize()
    for k in range(6):
        for i in (0, 1):
            g.assemble_vie(1.0, mats[i], out[i][k], stream=streams[i])
    torch.cuda.synchronize()
    for i in (0, 1):
        for M in out[i]:
            assert torch.equal(M, ref[i])
