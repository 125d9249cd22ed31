"""Assemblies of one geometry with different materials and frequencies on two
streams and from two threads: the geometry's Gram blocks and moment table serve
them in turn."""
import threading

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


@pytest.mark.parametrize("threads", [False, True])
def test_two_streams_two_frequencies(bfa, torch_cuda, threads):
    torch = torch_cuda
    V, T = kuhn(bfa, 5)
    g = bfa.Geometry(V, T)
    g.upload()
    g.build_static(6)
    mat = bfa.material("iso", eps=4 + 0.1j)
    new = lambda: torch.zeros((g.N, g.N), dtype=torch.complex128, device="cuda:0")
    calls = [lambda M, s=None: g.assemble_vie(1.0, mat, M, stream=s),
             lambda M, s=None: g.assemble_vie(2.5, mat, M, stream=s, far32=True)]
    ref = [new(), new()]
    for f, r in zip(calls, ref):
        f(r)
        torch.cuda.synchronize()
    assert (ref[0] - ref[1]).abs().max() > 0
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    out = [[new() for _ in range(6)] for _ in calls]
    torch.cuda.synchronize()
    if threads:
        def work(i):
            for M in out[i]:
                calls[i](M, streams[i])
        ts = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    else:
        for k in range(6):
            for i in (0, 1):
                calls[i](out[i][k], streams[i])
    torch.cuda.synchronize()
    for i in (0, 1):
        for M in out[i]:
            assert torch.equal(M, ref[i])
