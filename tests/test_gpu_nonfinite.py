"""GPU: diffusion sub-steps in which a concentration, a phase's share of it or a constant is not finite:
infinities and NaN stand where the full-formula kernel has them.  There an absent phase's partition is
0; the oracle divides for absent phases too, so its 0 * (inf - c) is NaN where the kernels have 0."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch  # before the library: both then use one HIP runtime

import oracle
from phasefield_amd import Domain, gpu_cleanup, gpu_diffusion_solver, lib
from phasefield_amd._capi import PfParams
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def params(tmp_path_factory):
    m = helpers.small_model(str(tmp_path_factory.mktemp("nf")), "fec_3d_256", nx=16, ny=16, nz=16,
                            grains=4, nuclei=2)
    q = oracle.as_orc_params(helpers.model_params(m))
    q.diffusivity[0][2] = 5.0
    return q


def ferrite(nx, ny, mixed_cells):
    """Ferrite with half austenite in `mixed_cells`: these and their neighbours take the full formula."""
    n = nx * ny
    ids, val, phase = np.zeros((n, 4), np.int32), np.zeros((n, 4)), np.zeros((n, 3))
    ids[:, 0], val[:, 0], phase[:, 1] = 200001, 1.0, 1.0
    for c in mixed_cells:
        ids[c, :2], val[c, :2], phase[c, :2] = (100001, 200001), 0.5, 0.5
    conc = 0.02 + 0.8 * np.random.default_rng(21).random(n)
    return ids.reshape(-1), val.reshape(-1), phase.reshape(-1), conc


def different(a, b):
    return np.flatnonzero(~((a == b) | (np.isnan(a) & np.isnan(b)))).tolist()


@pytest.mark.parametrize("form", [oracle.ORC_FP64, oracle.ORC_MIXED])
@pytest.mark.parametrize("P", [2, 3])
@pytest.mark.parametrize("count", [1, 3])
def test_overflowed_bulk_neighbour(P, form, count, params, monkeypatch):
    """A listed cell next to a bulk cell of infinite concentration."""
    print(f"[gpu] overflowed bulk neighbour P={P} form={form} count={count}", flush=True)
    nx, ny = 40, 24
    state = ferrite(nx, ny, [10 + nx * 10])
    state[3][8 + nx * 10] = np.inf  # bulk; its neighbour at x = 9 is listed
    q = PfParams.from_buffer_copy(params)
    q.dims = 2
    conc = []
    for kernel in ("lds", "bulk"):
        monkeypatch.setenv("PFAMD_DIFF_KERNEL", kernel)
        g = Domain(nx, ny, 1, depth=4, nphase=P,
                   precision="mixed" if form == oracle.ORC_MIXED else "fp64")
        g.set_params(q)
        g.upload(*state)
        g.diffuse(0, count, q.dt_d[0])
        conc.append(g.download()["conc"])
        g.close()
    assert np.isinf(conc[0]).any() and np.isnan(conc[0]).any() and np.isfinite(conc[0]).any()
    assert different(conc[1], conc[0]) == []


@pytest.mark.parametrize("loops", [1, 3])
def test_overflowed_partition_of_a_plane_with_six_faces(loops, params):
    """The accelerator calls sum six faces also where z is one cell: a phase whose partitioned
    concentration overflows gives inf - inf on the faces that join the cell to itself."""
    print(f"[gpu] overflowed partition, six faces, loops={loops}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    nx, ny = 40, 24
    cell = 10 + nx * 10
    ids, val, phase, conc = ferrite(nx, ny, [cell, cell - 1, cell + 1, cell - nx, cell + nx])
    conc[cell] = 1.5e308
    q = PfParams.from_buffer_copy(params)
    q.dims = 3
    q.part_k[0][0][1] = 0.1  # austenite's partition of the cell: c / 0.55
    D = np.array([q.diffusivity[0][i] for i in range(3)])
    pk = np.array([[q.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[q.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    dt = (loops - 0.1) * (q.dx * q.dx / D.max() / 2 * float(np.float32(0.2)))
    o = oracle.OracleDomain(nx, ny, 1, 4, 1)
    o.set_params(oracle.as_orc_params(q))
    o.set_state(ids, val, phase, conc)
    o.diffuse_factor(0, loops, dt / loops / (q.dx * q.dx))
    want = o.get_state()["conc"]
    assert np.isnan(want[cell]) and np.isfinite(want).any()
    host = conc.copy()
    gpu_diffusion_solver(D, pk, pc, phase, host, nx, ny, 1, dt, q.dx)
    gpu_cleanup()
    dphase = torch.from_numpy(phase).to("cuda:0")
    dconc = torch.from_numpy(conc).to("cuda:0")
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, dphase.data_ptr(), dconc.data_ptr(), nx, ny, 1, dt,
                                               q.dx, stream)
    assert rc == 0, lib().pf_last_error(None)
    assert different(dconc.cpu().numpy(), want) == []
    assert different(host, want) == []


@pytest.mark.parametrize("constant", ["D", "pk", "pc"])
@pytest.mark.parametrize("shape", [(40, 24, 1), (41, 24, 16)])
def test_nonfinite_constant_of_an_absent_phase(shape, constant, params):
    """The allocation-free call: a phase that no cell has, with a constant that is not finite, makes every
    cell NaN (0 * NaN), bulk cells too."""
    print(f"[gpu] non-finite {constant} {shape}", flush=True)
    nx, ny, nz = shape
    planes = [ferrite(nx, ny, [10 + nx * 10]) for _ in range(nz)]
    ids, val, phase, conc = (np.concatenate(a) for a in zip(*planes))
    q = PfParams.from_buffer_copy(params)
    q.dims = 3 if nz > 1 else 2
    D = np.array([q.diffusivity[0][i] for i in range(3)])
    dt = 2.9 * (q.dx * q.dx / D.max() / q.dims * float(np.float32(0.2)))
    if constant == "D":
        q.diffusivity[0][2] = D[2] = np.nan
    elif constant == "pk":
        q.part_k[0][1][2] = np.inf
    else:
        q.part_c[0][1][2] = np.inf
    pk = np.array([[q.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[q.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    o = oracle.OracleDomain(nx, ny, nz, 4, 1)
    o.set_params(oracle.as_orc_params(q))
    o.set_state(ids, val, phase, conc)
    o.diffuse_factor(0, 3, dt / 3 / (q.dx * q.dx))
    want = o.get_state()["conc"]
    assert np.isnan(want).all()
    dphase = torch.from_numpy(phase).to("cuda:0")
    dconc = torch.from_numpy(conc).to("cuda:0")
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, dphase.data_ptr(), dconc.data_ptr(), nx, ny, nz, dt,
                                               q.dx, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib().pf_last_error(None)
    assert different(dconc.cpu().numpy(), want) == []
