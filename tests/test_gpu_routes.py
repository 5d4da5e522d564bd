"""GPU: the diffusion kernels that the default rules do not pick at the tests' sizes, on the cases of
the other files: the plane-marching kernel (large 3D domains), the single sub-steps of planes, and the
adjoint over them.  The marching shape, which only that kernel sets, says which route a domain took."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch  # before the library: both then use one HIP runtime

import oracle
from phasefield_amd import Domain, gpu_cleanup, gpu_diffusion_solver, lib
from phasefield_amd._capi import PfParams
from tests import test_gpu_adjoint as adj
from tests import test_gpu_parity as par
from tests import test_gpu_substep_kernels as sub
from tests.test_gpu_parity import base_params  # noqa: F401  (fixture)
from tests.test_gpu_substep_kernels import params  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

FORMS = [oracle.ORC_FP64, oracle.ORC_MIXED]


@pytest.fixture
def shapes(monkeypatch):
    """The marching shapes of the domains of a test, when they end or have run the adjoint."""
    seen = []
    close, adjoint = Domain.close, Domain.adjoint

    def noted_close(self):
        if getattr(self, "_h", None):
            seen.append(self.march_shape())
        close(self)

    def noted_adjoint(self, *a, **k):
        r = adjoint(self, *a, **k)
        seen.append(self.march_shape())
        return r

    monkeypatch.setattr(Domain, "close", noted_close)
    monkeypatch.setattr(Domain, "adjoint", noted_adjoint)
    return seen


@pytest.fixture(params=["march", "default"])
def route(request, monkeypatch, shapes):
    """Run on the marching kernel and on the kernel of the default rules; the test ends with the check
    that it did."""
    if request.param == "march":
        monkeypatch.setenv("PFAMD_DIFF_DIRECT", "0")
        monkeypatch.setenv("PFAMD_DIFF_TILE", "off")
    yield request.param
    assert shapes
    for rows, zchunk in shapes:
        assert (rows > 0 and zchunk > 0) == (request.param == "march"), (rows, zchunk)


@pytest.fixture
def single(monkeypatch):
    monkeypatch.setenv("PFAMD_DIFF_DIRECT", "0")
    monkeypatch.setenv("PFAMD_DIFF_TILE", "off")


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("gamma_cols", [48, 16, 0])
def test_bulk_phase_choice(route, base_params, rng, form, gamma_cols):  # noqa: F811
    par.test_bulk_phase_choice_bitwise(base_params, rng, form, gamma_cols)


@pytest.mark.parametrize("form", FORMS)
def test_seeded_steps(route, tmp_path, monkeypatch, form):
    par.test_diffusion_kernel_variants_bitwise(tmp_path, monkeypatch, "bulk", "-1", "1", "1", "1", "0", form)


@pytest.mark.parametrize("form", FORMS)
def test_seeded_steps_noflux(route, tmp_path, monkeypatch, form):
    par.test_march_noflux_bitwise(tmp_path, monkeypatch, "-1", "0", form)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("bc", [0, 1])
def test_list_length(route, tmp_path, form, bc):
    par.test_diffusion_list_length(tmp_path, form, bc)


@pytest.mark.parametrize("form", FORMS)
def test_bulk_mask_change(route, tmp_path, form):
    par.test_bulk_mask_change_between_steps(tmp_path, form)


@pytest.mark.parametrize("shape,bc", [((33, 20, 12), 0), ((35, 18, 1), 0), ((41, 16, 10), 1)])
def test_mixed_listed_pass_odd_nx(single, tmp_path, shape, bc):
    par.test_mixed_listed_pass_odd_nx_bitwise(tmp_path, shape, bc)


@pytest.mark.parametrize("shape,bc", par.SHAPES)
@pytest.mark.parametrize("P", [2, 3])
def test_single_substeps(single, shape, bc, P, base_params, rng):  # noqa: F811
    par.test_diffusion_substeps_bitwise(shape, bc, P, base_params, rng)


@pytest.mark.parametrize("shape,bc", par.SHAPES)
def test_single_mixed_steps(single, shape, bc, base_params, rng):  # noqa: F811
    par.test_mixed_steps_random_states_bitwise(shape, bc, 4, 3, base_params, rng)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape,bc", [((2, 2, 2), 1), ((4, 4, 2), 1), ((2, 6, 1), 0), ((8, 2, 3), 0)])
def test_single_tiny_domains(single, shape, bc, form, base_params, rng):  # noqa: F811
    par.test_tiny_domains_bitwise(shape, bc, form, base_params, rng)


@pytest.mark.parametrize("shape,bc,K,P", [((20, 16, 12), "periodic", 4, 2), ((18, 14, 10), "noflux", 4, 3)])
def test_adjoint_gradients(route, tmp_path, monkeypatch, shape, bc, K, P):
    adj.test_adjoint_matches_dual_numbers(tmp_path, monkeypatch, shape, bc, K, P, "1")


@pytest.mark.parametrize("rows,bc", [("8", "periodic"), ("16", "noflux"), ("32", "periodic")])
def test_adjoint_gradients_by_tile_rows(tmp_path, monkeypatch, shapes, rows, bc):
    monkeypatch.setenv("PFAMD_DIFF_BY", rows)
    adj.test_adjoint_matches_dual_numbers(tmp_path, monkeypatch, (20, 16, 12), bc, 4, 2, "1")
    assert shapes and all(s[0] == int(rows) for s in shapes)


def test_adjoint_gradients_odd_nx(single, tmp_path, monkeypatch):
    adj.test_adjoint_matches_dual_numbers(tmp_path, monkeypatch, (21, 16, 10), "periodic", 4, 2, "1")


def test_adjoint_central_differences(route, tmp_path):
    adj.test_adjoint_matches_central_differences(tmp_path)


@pytest.mark.parametrize("shape,steps,every", [((20, 18, 10), 3, 2), ((40, 21, 1), 3, 3)])
def test_adjoint_state(single, shape, steps, every, params):  # noqa: F811
    sub.test_adjoint_leaves_the_stepped_state(shape, steps, every, params)


# ---- longer lists, larger planes ---------------------------------------------------------------------
def dense_state(rng, n, P):
    """Every cell of two phases: every cell is listed."""
    ids, val, phase = np.zeros((n, 4), np.int32), np.zeros((n, 4)), np.zeros((n, 3))
    w = 0.1 + 0.8 * rng.random(n)
    other = np.where(rng.random(n) < 0.3, 2, 1) if P == 3 else np.ones(n, int)
    ids[:, 0], ids[:, 1] = 100001, np.where(other == 2, 300001, 200001)
    val[:, 0], val[:, 1] = w, 1.0 - w
    phase[:, 0] = w
    phase[np.arange(n), other] = 1.0 - w
    return ids.reshape(-1), val.reshape(-1), phase.reshape(-1), 0.02 + 0.8 * rng.random(n)


LONG = [((40, 36, 30), 0, 2), ((65, 61, 39), 1, 3), ((104, 102, 100), 0, 2)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape,bc,P", LONG)
def test_more_listed_cells_than_threads(shape, bc, P, form, params):  # noqa: F811
    """Lists that go on behind the one-launch kernel's first workgroups, 16384 entries here: in the
    workgroups behind the bulk cells, in a second round of both (above 131072 entries), and, above 2^20
    cells, in rounds of the first alone; cells and byte pairs."""
    print(f"[gpu] long list {shape} bc={bc} P={P} form={form}", flush=True)
    n = int(np.prod(shape))
    sub.check(shape, bc, P, form, dense_state(np.random.default_rng(41), n, P), params, (1, 2))


@pytest.mark.parametrize("shape,bc,P", LONG)
def test_adjoint_more_listed_cells_than_threads(monkeypatch, shape, bc, P, params):  # noqa: F811
    """The reverse sub-step over the same lists, in one launch and in the separate listed pass: d_conc0
    by the same operations, the sums over the cells in another order."""
    print(f"[gpu] adjoint, long list {shape} bc={bc} P={P}", flush=True)
    q = PfParams.from_buffer_copy(params)
    q.n_sub[0] = 4
    n = int(np.prod(shape))
    state = dense_state(np.random.default_rng(42), n, P)
    r = []
    for direct in ("1", "0"):
        monkeypatch.setenv("PFAMD_DIFF_DIRECT", direct)
        g = Domain(*shape, depth=4, nphase=P, bc_z=bc)
        g.set_params(q)
        g.upload(*state)
        r.append(g.adjoint(1, [1], [0.3], 1.0, state[3] * 1.1))
        g.close()
    assert r[0]["loss"] == r[1]["loss"]
    assert np.abs(r[0]["d_conc0"]).max() > 0
    assert np.array_equal(r[0]["d_conc0"], r[1]["d_conc0"])
    for key in ("d_mobility", "d_sigma", "d_diff_gamma"):
        # n terms of either sign, summed in two orders: n * 2^-53 of the sum of their magnitudes,
        # which may exceed the sum by a factor of 1e3
        assert abs(r[0][key] - r[1][key]) <= n * 2.0 ** -53 * 1e3 * abs(r[1][key]), key


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("P", [2, 3])
def test_larger_plane(P, form, params):  # noqa: F811
    """Just above the plane size at which tiles grow to 32 x 32 cells, with odd extents."""
    shape = (363, 367, 1)
    print(f"[gpu] plane {shape} P={P} form={form}", flush=True)
    rng = np.random.default_rng(43)
    sub.check(shape, 0, P, form, sub.sparse_state(rng, *shape, P), params, (1, 14))
    for phases in range(2, P + 1):
        sub.check(shape, 0, P, form, dense_state(rng, 363 * 367, phases), params, (7,))


@pytest.mark.parametrize("shape", [(64, 33, 1), (37, 20, 11), (64, 12, 16), (363, 367, 1), (2, 200000, 1),
                                   (1300, 1161, 1)])
@pytest.mark.parametrize("loops", [1, 2])
def test_accelerator_calls_against_the_oracle(shape, loops, params):  # noqa: F811
    """Both accelerator calls, which share kernels, against the oracle, with few and with all cells
    listed: tiles, the one-launch kernel, and planes that take neither size of tile (narrow, and above
    1.5 M cells)."""
    print(f"[gpu] accelerator calls {shape} loops={loops}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    q = PfParams.from_buffer_copy(params)
    q.dims = 3  # six faces on every domain
    D = np.array([q.diffusivity[0][i] for i in range(3)])
    pk = np.array([[q.part_k[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    pc = np.array([[q.part_c[0][i][j] for j in range(3)] for i in range(3)]).T.reshape(-1).copy()
    dt = (loops - 0.1) * (q.dx * q.dx / D.max() / (3 if shape[2] > 1 else 2) * float(np.float32(0.2)))
    rng = np.random.default_rng(44)
    state = sub.sparse_state(rng, *shape, 3) if loops == 1 else dense_state(rng, int(np.prod(shape)), 2)
    o = oracle.OracleDomain(*shape, 4, 1)
    o.set_params(oracle.as_orc_params(q))
    o.set_state(*state)
    o.diffuse_factor(0, loops, dt / loops / (q.dx * q.dx))
    want = o.get_state()["conc"]
    host = state[3].copy()
    gpu_diffusion_solver(D, pk, pc, state[2], host, *shape, dt, q.dx)
    gpu_cleanup()
    assert np.flatnonzero(host != want)[:20].tolist() == []
    dphase, dconc = (torch.from_numpy(a).to("cuda:0") for a in state[2:])
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (D, pk, pc)]
    rc = lib().pf_gpu_diffusion_solver_noalloc(*ptr, dphase.data_ptr(), dconc.data_ptr(), *shape, dt,
                                               q.dx, stream)
    assert rc == 0, lib().pf_last_error(None)
    assert np.flatnonzero(dconc.cpu().numpy() != want)[:20].tolist() == []


@pytest.mark.parametrize("shape,pins,kernel,substeps", [
    ((64, 48, 1), {}, "diffuse_tile_kernel", 6),  # 20 sub-steps as 7 + 7 + 6
    ((64, 20, 12), {}, "diffuse_direct_kernel", 1),
    ((300, 1, 300), {}, "diffuse_bulk_march_kernel", 1),
    ((64, 20, 12), {"PFAMD_DIFF_DIRECT": "0"}, "diffuse_bulk_march_kernel", 1),
    ((33, 20, 12), {"PFAMD_DIFF_DIRECT": "0"}, "diffuse_linear_kernel", 1),
    ((64, 20, 12), {"PFAMD_DIFF_MARCH": "0"}, "diffuse_bulk_vec_kernel", 1),
    ((64, 20, 12), {"PFAMD_DIFF_VEC": "0", "PFAMD_DIFF_BY": "4"}, "diffuse_bulk_kernel", 1),
    ((64, 20, 12), {"PFAMD_DIFF_KERNEL": "lds"}, "diffuse_kernel", 1)])
def test_substep_kernel_is_named(monkeypatch, shape, pins, kernel, substeps, params):  # noqa: F811
    print(f"[gpu] sub-step kernel of {shape} {pins}", flush=True)
    for k, v in pins.items():
        monkeypatch.setenv(k, v)
    q = PfParams.from_buffer_copy(params)
    q.dims = 3 - (shape[2] == 1) - (shape[1] == 1)
    g = Domain(*shape, depth=4)
    g.set_params(q)
    g.upload(*sub.sparse_state(np.random.default_rng(45), *shape, 2))
    assert g.substep_kernel() == (None, 0)
    g.diffuse(0, 20, q.dt_d[0])
    assert g.substep_kernel() == (kernel, substeps)
    g.close()
