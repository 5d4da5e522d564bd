"""GPU: the diffusion sub-step kernels at the sizes where they can go wrong, bitwise against the
oracle: rows of every remainder, odd plane counts, extents that wrap onto themselves, insulated z,
every phase count and both forms, each on random states (nearly every cell listed) and on states
that are bulk but for a few cells.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from phasefield_amd import Domain
from phasefield_amd._capi import PfParams
from tests import helpers

pytestmark = pytest.mark.gpu

FORMS = [oracle.ORC_FP64, oracle.ORC_MIXED]


@pytest.fixture(scope="module")
def params(tmp_path_factory):
    m = helpers.small_model(str(tmp_path_factory.mktemp("sk")), "fec_3d_256", nx=16, ny=16, nz=16,
                            grains=4, nuclei=2)
    q = oracle.as_orc_params(helpers.model_params(m))
    q.diffusivity[0][2] = 5.0
    return q


def sparse_state(rng, nx, ny, nz, P):
    """Ferrite with a slab of austenite and some mixed cells: bulk cells of both phases and a list."""
    n = nx * ny * nz
    ids, val = np.zeros((n, 4), np.int32), np.zeros((n, 4))
    phase = np.zeros((n, 3))
    gamma = np.arange(n) % nx < nx // 3
    ids[:, 0] = np.where(gamma, 100001, 200001)
    val[:, 0] = 1.0
    phase[:, 0], phase[:, 1] = gamma, ~gamma
    some = rng.choice(n, size=max(1, n // 40), replace=False)
    w = 0.1 + 0.8 * rng.random(some.size)
    ids[some, 0], ids[some, 1] = 100001, 200001
    val[some, 0], val[some, 1] = w, 1.0 - w
    phase[some] = 0.0
    phase[some, 0], phase[some, 1] = w, 1.0 - w
    if P == 3:
        one = some[0]
        ids[one, 0], val[one, 0], phase[one, 0], phase[one, 2] = 300001, w[0], 0.0, w[0]
    return ids.reshape(-1), val.reshape(-1), phase.reshape(-1), 0.02 + 0.8 * rng.random(n)


def check(shape, bc, P, form, state, params, counts):
    nx, ny, nz = shape
    q = PfParams.from_buffer_copy(params)
    q.dims = 3 - (nz == 1) - (ny == 1)
    g = Domain(nx, ny, nz, depth=4, nphase=P, precision="mixed" if form == oracle.ORC_MIXED else "fp64",
               bc_z=bc)
    g.set_params(q)
    g.upload(*state)
    o = oracle.OracleDomain(nx, ny, nz, 4, 1, form, bc)
    o.set_params(oracle.as_orc_params(q))
    o.set_state(*state)
    for n in counts:
        g.diffuse(0, n, q.dt_d[0])
        o.diffuse(0, n, q.dt_d[0])
    a, b = g.download(), o.get_state()
    g.close()
    assert np.array_equal(a["conc"], b["conc"])
    if form == oracle.ORC_MIXED:
        assert np.array_equal(a["conc_comp"], b["conc_comp"])


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape,bc,P", [((64, 20, 9), 0, 2), ((66, 7, 8), 1, 2), ((67, 9, 11), 0, 3),
                                        ((33, 5, 3), 1, 2), ((128, 4, 2), 0, 3), ((3, 2, 5), 0, 2),
                                        ((2, 3, 2), 1, 2), ((131, 6, 7), 1, 3)])
def test_one_launch_substep_bitwise(shape, bc, P, form, params):
    print(f"[gpu] one-launch sub-step {shape} bc={bc} P={P} form={form}", flush=True)
    rng = np.random.default_rng(11)
    check(shape, bc, P, form, sparse_state(rng, *shape, P), params, (1, 4))
    ids, val, phase, conc = helpers.random_state(rng, *shape, 4, nphase=P)
    check(shape, bc, P, form, (ids, val, phase, conc), params, (3,))


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape,P,pin", [((64, 48, 1), 2, ""), ((61, 47, 1), 2, "20,18,12"),
                                         ((61, 47, 1), 3, "16,16,12"), ((130, 9, 1), 2, "16,16,5"),
                                         ((5, 4, 1), 2, "16,16,12"), ((2, 3, 1), 3, ""),
                                         ((40, 1, 13), 2, "16,16,4"), ((400, 30, 1), 2, "")])
def test_many_substeps_per_launch_bitwise(shape, P, pin, form, params, monkeypatch):
    """Tiles whose halo is narrower and wider than the domain, partial last tiles, sub-step counts that
    do not divide, tiles that are nearly all bulk and tiles with more listed cells than entries."""
    print(f"[gpu] tiles {shape} P={P} pin={pin} form={form}", flush=True)
    monkeypatch.setenv("PFAMD_DIFF_TILE", pin)
    rng = np.random.default_rng(12)
    check(shape, 0, P, form, sparse_state(rng, *shape, P), params, (1, 25))
    ids, val, phase, conc = helpers.random_state(rng, *shape, 4, nphase=P)
    check(shape, 0, P, form, (ids, val, phase, conc), params, (13,))


@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("shape", [(64, 33, 1), (5, 7, 1), (37, 20, 11), (64, 12, 16), (2, 2, 2)])
def test_noalloc_kernels_bitwise(shape, skip, params):
    """The allocation-free call on its tile and one-launch kernels, on arrays that are aligned to 16
    bytes and to one value only, twice in a row, against the call on host buffers."""
    import ctypes

    import torch

    from phasefield_amd import gpu_cleanup, gpu_diffusion_solver, lib
    print(f"[gpu] noalloc kernels {shape} skip={skip}", flush=True)
    rng = np.random.default_rng(13)
    n = int(np.prod(shape))
    D = np.array([params.diffusivity[0][i] for i in range(3)])
    pk = np.array([[params.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[params.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    dt = 0.11 * params.pfm_dt
    for state in (sparse_state(rng, *shape, 2), helpers.random_state(rng, *shape, 4)):
        phase, conc = state[2], state[3]
        dphase = torch.zeros(3 * n + skip, dtype=torch.float64, device="cuda:0")[skip:]
        dconc = torch.zeros(n + skip, dtype=torch.float64, device="cuda:0")[skip:]
        dphase.copy_(torch.from_numpy(phase))
        dconc.copy_(torch.from_numpy(conc))
        ref = conc.copy()
        for _ in range(2):
            gpu_diffusion_solver(D, pk, pc, phase, ref, *shape, dt, params.dx)
            rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, dphase.data_ptr(), dconc.data_ptr(), *shape,
                                                       dt, params.dx,
                                                       torch.cuda.current_stream().cuda_stream)
            assert rc == 0, lib().pf_last_error(None)
        assert np.array_equal(dconc.cpu().numpy(), ref)
    gpu_cleanup()


@pytest.mark.parametrize("shape,steps,every", [((20, 18, 10), 1, 1), ((20, 18, 10), 3, 2),
                                               ((33, 9, 7), 5, 3), ((40, 21, 1), 3, 3)])
def test_adjoint_leaves_the_stepped_state(shape, steps, every, params):
    """The steps whose sub-steps are kept as they run leave what plain steps leave: the checkpoint
    (state and sub-step counter) and the step after it; a run that recomputes every step from its
    checkpoints gives the same gradients."""
    print(f"[gpu] adjoint state {shape} steps={steps} every={every}", flush=True)
    nx, ny, nz = shape
    q = PfParams.from_buffer_copy(params)
    q.dims = 3 - (nz == 1)
    q.n_sub[0] = 7
    state = sparse_state(np.random.default_rng(14), *shape, 2)
    blob, grad = [], []
    for mode in ("plain", "segment", "step"):
        g = Domain(nx, ny, nz, depth=4)
        g.set_params(q)
        g.upload(*state)
        if mode == "plain":
            g.step(steps)
        else:
            with pytest.MonkeyPatch.context() as mp:
                mp.setenv("PFAMD_ADJ_RECOMPUTE", mode)
                grad.append(g.adjoint(steps, [steps], [0.3], checkpoint_every=every))
        a = g.checkpoint()
        g.step(1)
        blob.append((a, g.download()["conc"]))
        g.close()
    assert blob[0][0] == blob[1][0]
    for _, conc in blob[1:]:
        assert np.array_equal(conc, blob[0][1])
    for key in ("loss", "d_mobility", "d_sigma", "d_diff_gamma"):
        assert grad[0][key] == grad[1][key], key
    assert np.array_equal(grad[0]["d_conc0"], grad[1]["d_conc0"])
