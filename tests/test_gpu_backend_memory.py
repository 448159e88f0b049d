"""GPU: the Exec mirror where device memory is short -- images that the card or
the budget has no room for, and what is asked for after them."""
import ctypes

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


def test_images_make_way_for_later_weights(gpu, oracle, backend):
    """Under a budget that the first weight's images fill, a second weight, a
    scratch and a buffer are still placed; products read what is left."""
    tt, rows, cols, tokens = po.TT_Q5_K, 2048, 5120, 40
    ws = [synth.make_weight(tt, rows, cols, seed=65 + i, tag=tt) for i in range(3)]
    budget = 9 * rows * cols // 2  # six weights' bytes, or one weight and its images
    backend.set_mem_budget(budget)
    lins = [backend.load_linear(tt, rows, cols, ws[0])]
    assert backend.prepare_linear(lins[0]) == 0
    assert backend.mem_placed() > 4 * rows * cols  # no room beside them
    lins += [backend.load_linear(tt, rows, cols, w) for w in ws[1:]]
    buf = ctypes.c_void_p()
    assert backend.lib.qhip_backend_alloc_buf(backend._h, rows * cols // 8, ctypes.byref(buf)) == 0 and buf.value
    for lin, w in zip(lins, ws):
        for k in (1, tokens):
            x = synth.make_act(cols, k, seed=68)
            out = torch.empty((k, rows), device=gpu)
            backend.matvec_batch_k(out, lin, torch.from_numpy(x).to(gpu), k)
            assert rel_l2(out.cpu().numpy(), oracle.matvec(tt, w, x)) < TOL
    assert backend.mem_placed() <= budget


def test_captured_images_stay(gpu, oracle, backend):
    """A graph captured from an image keeps it: a load that would need its room
    is refused, and the graph replays on."""
    tt, rows, cols = po.TT_Q5_K, 512, 5120
    w = synth.make_weight(tt, rows, cols, seed=69, tag=tt)
    lin = backend.load_linear(tt, rows, cols, w)
    assert backend.prepare_linear(lin) == 0
    x, out = torch.empty((1, cols), device=gpu), torch.empty((1, rows), device=gpu)
    side = torch.cuda.Stream()
    backend.set_stream(side)
    backend.matvec(out, lin, x)  # the scratch
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        backend.matvec(out, lin, x)
    placed = backend.mem_placed()
    backend.set_mem_budget(placed + 1024)
    with pytest.raises(Exception):
        backend.load_linear(tt, rows, cols, w)
    assert backend.mem_placed() == placed
    for i in range(3):
        xi = synth.make_act(cols, 1, seed=70 + i)
        x.copy_(torch.from_numpy(xi))
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy(), oracle.matvec(tt, w, xi)) < TOL
