"""GPU: the Exec mirror where device memory is short -- images that the card or
the budget has no room for, and what is asked for after them."""
import numpy as np
import pytest
import torch

import pyoracle as po
from qwen35_amd import _lib, ops, synth

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


@pytest.mark.parametrize("tt", [po.TT_Q5_K, po.TT_Q3_K, po.TT_IQ4_XS])
def test_refused_image_leaves_no_error(gpu, oracle, backend, tt):
    """Images larger than the card are refused when the weight is prepared, and
    the products that follow on this thread still succeed."""
    rows, cols, few = 64, 5120, 40
    w = synth.make_weight(tt, rows, cols, seed=61, tag=tt)
    lin = backend.load_linear(tt, rows, cols, w)
    # a handle alone: nothing is read through it, for no image is allocated
    huge = _lib.QhipLinear(lin.dev, tt, 1 << 26, 17408, _lib.load().qhip_weight_row_bytes(tt, 17408))
    placed = backend.mem_placed()
    assert backend.prepare_linear(huge) == -1 and backend.mem_placed() == placed
    for tokens in (1, few):
        x = synth.make_act(cols, tokens, seed=62)
        out = torch.empty((tokens, rows), device=gpu)
        backend.matvec_batch_k(out, lin, torch.from_numpy(x).to(gpu), tokens)
        assert rel_l2(out.cpu().numpy(), oracle.matvec(tt, w, x)) < TOL
    assert backend.prepare_linear(lin) == 0  # a refusal is not kept against a smaller image


# a prompt from the plane image, and one token from a GEMV image
@pytest.mark.parametrize("tt,rows,cols,tokens", [(po.TT_Q3_K, 300, 1024, 140), (po.TT_Q6_K, 300, 1024, 140),
                                                 (po.TT_Q5_K, 300, 9728, 1), (po.TT_IQ4_NL, 2049, 5120, 1)])
def test_image_leaves_room_for_the_activations(gpu, oracle, backend, tt, rows, cols, tokens):
    """A budget that holds the image or the activations, not both: the image is
    not built and the product runs from the GGUF rows."""
    w = synth.make_weight(tt, rows, cols, seed=63, tag=tt)
    x = synth.make_act(cols, tokens, seed=64)
    xd, out = torch.from_numpy(x).to(gpu), torch.empty((tokens, rows), device=gpu)
    lin = backend.load_linear(tt, rows, cols, w)
    base = backend.mem_placed()
    assert backend.prepare_linear(lin) == 0
    image = backend.mem_placed() - base
    assert image > 0
    again = ops.Backend(0)
    try:
        lin = again.load_linear(tt, rows, cols, w)
        again.set_mem_budget(again.mem_placed() + image + 512)
        for _ in range(2):
            out.fill_(float("nan"))
            again.matvec_batch_k(out, lin, xd, tokens)
            at = np.unique(np.r_[0:min(rows, 300), rows - 1])
            want = oracle.matvec(tt, np.ascontiguousarray(w.reshape(rows, -1)[at]), x)
            assert rel_l2(out.cpu().numpy()[:, at], want) < TOL
    finally:
        again.close()
