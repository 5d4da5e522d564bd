"""GPU: the accelerator calls (host buffers, and the allocation-free one) on domains of one row or one
column.  They sum six faces on every domain, also where a step of that domain has four."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch  # before the library: both then use one HIP runtime

import oracle
from phasefield_amd import gpu_cleanup, gpu_diffusion_solver, lib
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(48, 1, 20), (33, 1, 7), (1, 9, 8), (7, 1, 2)])
def test_six_faces_on_one_row(tmp_path, shape):
    print(f"[gpu] accelerator calls on {shape}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    m = helpers.small_model(str(tmp_path), "fec_3d_256", nx=16, ny=16, nz=16, grains=4, nuclei=2)
    q = oracle.as_orc_params(helpers.model_params(m))
    q.dims = 3
    D = np.array([q.diffusivity[0][i] for i in range(3)])
    pk = np.array([[q.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[q.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    loops = 5
    dt = (loops - 0.1) * (q.dx * q.dx / D.max() / (3 if shape[2] > 1 else 2) * float(np.float32(0.2)))
    ids, val, phase, conc = helpers.random_state(np.random.default_rng(31), *shape, 4)
    o = oracle.OracleDomain(*shape, 4, 1)
    o.set_params(q)
    o.set_state(ids, val, phase, conc)
    o.diffuse_factor(0, loops, dt / loops / (q.dx * q.dx))
    want = o.get_state()["conc"]
    host = conc.copy()
    gpu_diffusion_solver(D, pk, pc, phase, host, *shape, dt, q.dx)
    gpu_cleanup()
    assert np.flatnonzero(host != want).tolist() == []
    dphase = torch.from_numpy(phase).to("cuda:0")
    dconc = torch.from_numpy(conc).to("cuda:0")
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, dphase.data_ptr(), dconc.data_ptr(), *shape, dt,
                                               q.dx, stream)
    assert rc == 0, lib().pf_last_error(None)
    assert np.flatnonzero(dconc.cpu().numpy() != want).tolist() == []


@pytest.mark.parametrize("shape", [(37, 20, 11), (40, 24, 1), (48, 1, 20), (128, 90, 93)])
def test_no_phase_with_identity_partition(tmp_path, shape):
    """Tables without an identity partition, so that no cell has a reduced form, on states whose cells
    would all have one."""
    print(f"[gpu] no identity partition {shape}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    m = helpers.small_model(str(tmp_path), "fec_3d_256", nx=16, ny=16, nz=16, grains=4, nuclei=2)
    q = oracle.as_orc_params(helpers.model_params(m))
    q.dims = 3
    for p in range(3):
        q.part_k[0][p][p] = 1.1
    D = np.array([q.diffusivity[0][i] for i in range(3)])
    pk = np.array([[q.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[q.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    loops = 4
    dt = (loops - 0.1) * (q.dx * q.dx / D.max() / (3 if shape[2] > 1 else 2) * float(np.float32(0.2)))
    n = int(np.prod(shape))
    ids, val, phase = np.zeros((n, 4), np.int32), np.zeros((n, 4)), np.zeros((n, 3))
    gamma = np.arange(n) % shape[0] < shape[0] // 3
    ids[:, 0], val[:, 0] = np.where(gamma, 100001, 200001), 1.0
    phase[:, 0], phase[:, 1] = gamma, ~gamma
    phase[n // 2] = (0.4, 0.6, 0.0)
    phase, conc = phase.reshape(-1), 0.02 + 0.8 * np.random.default_rng(32).random(n)
    o = oracle.OracleDomain(*shape, 4, 1)
    o.set_params(q)
    o.set_state(ids.reshape(-1), val.reshape(-1), phase, conc)
    o.diffuse_factor(0, loops, dt / loops / (q.dx * q.dx))
    want = o.get_state()["conc"]
    host = conc.copy()
    gpu_diffusion_solver(D, pk, pc, phase, host, *shape, dt, q.dx)
    gpu_cleanup()
    assert np.flatnonzero(host != want).tolist() == []
    dphase = torch.from_numpy(phase).to("cuda:0")
    dconc = torch.from_numpy(conc).to("cuda:0")
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, dphase.data_ptr(), dconc.data_ptr(), *shape, dt,
                                               q.dx, stream)
    assert rc == 0, lib().pf_last_error(None)
    assert np.flatnonzero(dconc.cpu().numpy() != want).tolist() == []
