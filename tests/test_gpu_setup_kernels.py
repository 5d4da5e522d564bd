"""GPU: the seeded setup (tessellation with seeds dropped per block of cells, growth, nuclei with a
kept flag maximum per run of cells) bitwise against the oracle, at the sizes where it can go wrong:
blocks and runs that the domain does not fill, insulated z, more seeds than one pass takes, seeds outside the
domain, stretched distances, boxes that wrap or take whole axes, negative flags.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from phasefield_amd import Domain
from phasefield_amd._capi import PfParams
from tests import helpers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,depth,grains,reduction,nuclei,radius,conc,bc", [
    ((2, 2, 1), 4, 1, 0.0, 1, 1.0, 0.2, 0),
    ((5, 3, 2), 4, 4, 0.0, 3, 1.5, 0.2, 0),
    ((17, 33, 1), 4, 5, 0.0, 4, 3.0, 0.2, 0),
    ((130, 70, 1), 6, 300, 0.1, 9, 4.0, 3.5, 0),
    ((9, 7, 13), 4, 3, 0.2, 5, 40.0, 0.2, 0),
    ((64, 64, 3), 4, 20, 0.0, 8, 2.5, 0.2, 0),
    ((40, 23, 19), 6, 70, 0.0, 12, 3.0, 3.5, 0),
    ((33, 41, 29), 4, 600, 0.3, 20, 2.0, 0.2, 0),
    ((29, 31, 37), 4, 60, 0.0, 6, 2.0, 0.2, 1),
    # from 3 * 2^20 cells on the growth classifies copy cells and lists the others
    ((162, 141, 139), 4, 900, 0.0, 10, 3.0, 0.2, 0),
    ((149, 147, 146), 6, 900, 0.0, 10, 3.0, 3.5, 1),
    ((1801, 1771, 1), 4, 500, 0.1, 10, 5.0, 0.2, 0),
])
def test_setup_sizes(tmp_path, shape, depth, grains, reduction, nuclei, radius, conc, bc):
    nx, ny, nz = shape
    print(f"setup {shape} depth {depth} grains {grains} nuclei {nuclei} radius {radius} bc {bc}", flush=True)
    m = helpers.small_model(str(tmp_path), "fec_3d_256", nx=16, ny=16, nz=16, grains=4, nuclei=2)
    q = PfParams.from_buffer_copy(helpers.model_params(m))
    q.dims = 3 - (nz == 1) - (ny == 1)
    rng = np.random.default_rng(nx * 1000 + ny * 10 + nz)
    seeds = 0.5 + rng.random((grains, 3)) * np.array(shape)
    if grains > 4:  # two equal seeds, one outside of the domain
        seeds[3] = seeds[1]
        seeds[2] = [2.5 * nx, -3.0, 1.7 * nz]
    seeds = np.ascontiguousarray(seeds)
    g = Domain(nx, ny, nz, depth=depth, bc_z=bc)
    g.set_params(q)
    g.construct(seeds, reduction, 3, [conc] * 3)
    g.nucleate(nuclei, radius, (0.8, -1.0), 77)
    o = oracle.OracleDomain(nx, ny, nz, depth, 1, oracle.ORC_FP64, bc)
    o.set_params(oracle.as_orc_params(q))
    o.construct(oracle.tessellation(nx, ny, nz, seeds, reduction), 3, [conc] * 3)
    o.nucleate(nuclei, radius, (0.8, -1.0), 77)
    dev, ref = g.download(), o.get_state()
    for name in ("index", "value", "phase", "conc"):
        assert np.array_equal(dev[name], ref[name]), name
