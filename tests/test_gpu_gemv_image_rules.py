"""GPU: when a one-token product of the Exec mirror reads its weight's GEMV image
-- as one weight and as half of an adjacent pair, with the activation memo on,
and for an x that the one-launch form does not take."""
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


def load_pair(be, tt, rows, cols, seed):
    w = synth.make_weight(tt, 2 * rows, cols, seed=seed, tag=tt).reshape(2 * rows, -1)
    return w, [be.load_linear(tt, rows, cols, part) for part in (w[:rows], w[rows:])]


# every weight alone takes the one-launch form (Q3_K: too small for an image),
# the pair an image
@pytest.mark.parametrize("tt,rows,cols", [(po.TT_Q8_0, 4160, 4096), (po.TT_IQ4_NL, 4160, 4096),
                                          (po.TT_Q5_K, 16400, 2560), (po.TT_Q3_K, 1792, 2560)])
def test_prepared_pair_is_captured_from_its_images(gpu, oracle, backend, tt, rows, cols):
    w, (a, b) = load_pair(backend, tt, rows, cols, seed=71)
    assert backend.lib.qhip_backend_alloc_scratch(backend._h, cols) == 0
    assert backend.prepare_linear(a) == 0 and backend.prepare_linear(b) == 0
    placed = backend.mem_placed()
    x, out = torch.empty(cols, device=gpu), torch.empty(2 * rows, device=gpu)
    side = torch.cuda.Stream()
    backend.set_stream(side)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=side):
        backend.matvec_pair(out, a, b, x)
    backend.set_stream(torch.cuda.current_stream())
    eager = torch.empty_like(out)
    at = np.unique(np.linspace(0, 2 * rows - 1, 200).astype(int))
    for i in range(3):
        xi = synth.make_act(cols, 1, seed=72 + i)
        x.copy_(torch.from_numpy(xi[0]))
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy()[at], oracle.matvec(tt, np.ascontiguousarray(w[at]), xi)[0]) < TOL
        backend.matvec_pair(eager, a, b, x)
        assert torch.equal(out, eager)  # the same launch, so the graph reads the images too
    assert backend.mem_placed() == placed  # nothing was left to build


@pytest.mark.parametrize("cols", [2560, 4096])
@pytest.mark.parametrize("tt", [po.TT_Q8_0, po.TT_IQ4_NL, po.TT_Q4_0])
def test_memo_and_unaligned_x_read_the_image(gpu, oracle, backend, tt, cols):
    """Past 2^23 weights, where the one-launch form is the faster of the two: an x
    that it does not take, and one it has quantized already, are multiplied from
    the image."""
    rows = 3300
    w = synth.make_weight(tt, rows, cols, seed=75, tag=tt)
    lin = backend.load_linear(tt, rows, cols, w)
    base = backend.mem_placed()
    assert backend.prepare_linear(lin) == 0
    assert backend.mem_placed() > base
    x = synth.make_act(cols, 1, seed=76)
    buf = torch.empty(cols + 4, device=gpu)
    outs = {}
    for shift in (0, 1):  # floats past a 16-byte boundary
        xd = buf[shift:shift + cols]
        xd.copy_(torch.from_numpy(x[0]))
        for memo in (False, True):
            backend.set_act_memo(memo)
            for again in range(3):
                out = torch.empty(rows, device=gpu)
                backend.matvec(out, lin, xd)
                outs[shift, memo, again] = out
    want = oracle.matvec(tt, w, x)[0]
    for out in outs.values():
        assert rel_l2(out.cpu().numpy(), want) < TOL
    fused, image = outs[0, False, 0], outs[1, False, 0]
    # where a row's terms are summed in another order, the bits tell the two apart
    assert cols == 4096 or not torch.equal(fused, image)
    for (shift, memo, again), out in outs.items():
        # the one-launch form leaves the activation in the image's own layout
        from_image = shift == 1 or (memo and again > 0)
        assert torch.equal(out, image if from_image else fused), (shift, memo, again)
    assert backend.act_stats() == (4, 2)  # per x, the later products reuse the first one's activation


def test_memo_one_launch_rows_for_a_weight_without_image(gpu, oracle, backend):
    """Without an image the one-launch form leaves the reference rows, as for a
    weight too small for one, and the two kinds of one x do not meet."""
    tt, cols = po.TT_Q8_0, 2560
    ws = [synth.make_weight(tt, rows, cols, seed=79, tag=rows) for rows in (3300, 500)]
    large, small = (backend.load_linear(tt, w.reshape(-1, 2720).shape[0], cols, w) for w in ws)
    assert backend.prepare_linear(large) == 0
    x = synth.make_act(cols, 1, seed=80)
    xd = torch.from_numpy(x[0]).to(gpu)
    want = [oracle.matvec(tt, w, x)[0] for w in ws]
    backend.set_act_memo(True)
    for images in (True, False):
        backend.set_gemv_images(images)
        for lin, ref in ((large, 0), (large, 0), (small, 1), (small, 1), (large, 0), (large, 0), (small, 1)):
            out = torch.empty(lin.rows, device=gpu)
            backend.matvec(out, lin, xd)
            assert rel_l2(out.cpu().numpy(), want[ref]) < TOL


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
