"""GPU: the allocation-free diffusion call recorded into a graph, on each of its routes, replayed several
times with eager calls between the replays: every replay equals the eager result bit for bit."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch  # before the library: both then use one HIP runtime

import oracle
from phasefield_amd import lib
from tests import helpers

pytestmark = pytest.mark.gpu


# tiles; one launch (rows of whole runs, odd rows); above 2^20 cells; no identity partition there
@pytest.mark.parametrize("shape,identity", [((40, 24, 1), True), ((40, 24, 16), True), ((33, 21, 9), True),
                                            ((128, 90, 93), True), ((128, 90, 93), False)])
@pytest.mark.parametrize("loops", [2, 5])
def test_replays_equal_eager(tmp_path, shape, identity, loops):
    print(f"[gpu] capture {shape} identity={identity} loops={loops}", flush=True)
    m = helpers.small_model(str(tmp_path), "fec_3d_256", nx=16, ny=16, nz=16, grains=4, nuclei=2)
    q = oracle.as_orc_params(helpers.model_params(m))
    if not identity:
        for p in range(3):
            q.part_k[0][p][p] = 1.1
    D = np.array([q.diffusivity[0][i] for i in range(3)])
    pk = np.array([[q.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[q.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    dt = (loops - 0.1) * (q.dx * q.dx / D.max() / (3 if shape[2] > 1 else 2) * float(np.float32(0.2)))
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    n = int(np.prod(shape))
    phases, concs = [], []
    for seed in range(2):  # two phases side by side, a tenth of the cells mixed
        rng = np.random.default_rng(50 + seed)
        f = (np.arange(n) % shape[0] < shape[0] // (2 + seed)).astype(float)
        mixed = rng.random(n) < 0.1
        f[mixed] = rng.random(int(mixed.sum()))
        phases.append(torch.from_numpy(np.stack([f, 1 - f, 0 * f], 1).reshape(-1)).to("cuda:0"))
        concs.append(torch.from_numpy(0.02 + 0.8 * rng.random(n)).to("cuda:0"))
    phase, conc = phases[0].clone(), concs[0].clone()

    def call():
        rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, phase.data_ptr(), conc.data_ptr(), *shape, dt,
                                                   q.dx, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib().pf_last_error(None)

    def load(k):
        phase.copy_(phases[k])
        conc.copy_(concs[k])

    want = []
    for k in range(2):
        load(k)
        call()
        want.append(conc.clone())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for replay in range(4):
        k = replay % 2
        load(k)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(conc, want[k]), replay
        load(1 - k)  # an eager call on other values, in the same scratch
        call()
        torch.cuda.synchronize()
        assert torch.equal(conc, want[1 - k]), replay
