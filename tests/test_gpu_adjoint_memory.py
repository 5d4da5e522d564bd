"""GPU: the device memory that adjoint runs keep goes back when it is asked for and with its handle,
and the runs before and after give the same."""
from __future__ import annotations

import numpy as np
import pytest
import torch  # before the library: both then use one HIP runtime

from phasefield_amd import Domain, lib
from phasefield_amd._capi import PF_ERR_INVALID
from tests import helpers

pytestmark = pytest.mark.gpu


def test_kept_memory_goes_back(tmp_path):
    print("[gpu] adjoint memory", flush=True)
    m = helpers.small_model(str(tmp_path), "fec_3d_256", nx=64, ny=64, nz=64, grains=4, nuclei=3)
    p = helpers.model_params(m)
    p.n_sub[0] = 50
    ids, val, phase, conc = _ferrite(64 ** 3)
    g = Domain(64, 64, 64, depth=4)
    g.set_params(p)
    block = 100 << 20  # a step's 51 carbon fields alone are 107 MB
    free, runs = [], []

    def note():
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])

    def run():
        g.upload(ids, val, phase, conc)
        runs.append(g.adjoint(1, [1], [0.3]))

    note()
    g.adjoint_release()  # nothing kept yet
    run()
    note()
    g.adjoint_release()
    note()
    run()
    note()
    g.close()
    note()
    assert free[1] < free[0] - block
    assert free[2] > free[1] + block
    assert free[3] < free[2] - block
    assert free[4] > free[3] + block
    for key in ("loss", "d_mobility", "d_sigma", "d_diff_gamma"):
        assert runs[0][key] == runs[1][key], key
    assert np.array_equal(runs[0]["d_conc0"], runs[1]["d_conc0"])
    assert lib().pf_adjoint_release(None) == PF_ERR_INVALID


def _ferrite(n):
    ids, val, phase = np.zeros((n, 4), np.int32), np.zeros((n, 4)), np.zeros((n, 3))
    ids[:, 0], val[:, 0], phase[:, 1] = 200001, 1.0, 1.0
    some = np.random.default_rng(5).choice(n, size=n // 50, replace=False)
    ids[some, :2], val[some, :2], phase[some, :2] = (100001, 200001), 0.5, 0.5
    return ids.reshape(-1), val.reshape(-1), phase.reshape(-1), 0.02 + 0.5 * phase[:, 0]
