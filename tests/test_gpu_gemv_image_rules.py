"""GPU: when a one-token product of the Exec mirror reads its weight's GEMV
image."""
import numpy as np
import pytest
import torch

import pyoracle as po
from qwen35_amd import ops, synth

pytestmark = pytest.mark.gpu
TOL = 1e-5


def rel_l2(got, want):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    return float(np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30))


@pytest.fixture
def backend(gpu):
    be = ops.Backend(0)
    yield be
    be.close()


# one round of the one-launch form's workgroups | a little past it
@pytest.mark.parametrize("rows,cols,image", [(8192, 2560, False), (12800, 2560, True), (5120, 5120, True)])
def test_second_round_takes_the_image(gpu, oracle, backend, rows, cols, image):
    tt = po.TT_Q8_0
    w = synth.make_weight(tt, rows, cols, seed=77, tag=rows)
    lin = backend.load_linear(tt, rows, cols, w)
    placed = backend.mem_placed()
    x = synth.make_act(cols, 1, seed=78)
    out = torch.empty(rows, device=gpu)
    backend.matvec(out, lin, torch.from_numpy(x[0]).to(gpu))
    assert (backend.mem_placed() - placed > rows * cols) == image
    at = np.unique(np.linspace(0, rows - 1, 200).astype(int))
    want = oracle.matvec(tt, np.ascontiguousarray(w.reshape(rows, -1)[at]), x)[0]
    assert rel_l2(out.cpu().numpy()[at], want) < TOL
