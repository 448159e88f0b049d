"""GPU: the GEMV images of Q2_K, Q3_K and Q5_K (each unit's own bits), which the
Exec mirror reads at one token: every launch shape (two-wave teams, four-wave
teams, balanced teams of one and of four waves), row counts that are no multiple
of a team's rows and rows of fewer units than lanes, against the oracle and
against the GGUF rows; adjacent weights; a captured launch; and the public image
calls, which keep to their formats."""
import numpy as np
import pytest
import torch

import pyoracle as po
from qwen35_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu
FORMATS = [po.TT_Q2_K, po.TT_Q3_K, po.TT_Q5_K]
# two-wave teams | four-wave | balanced, one wave: b = 0, b = 16, b = 20 | more
# tail units than a wave takes (b = 36) | balanced, four waves
SHAPES = [(333, 5120), (5, 8192), (39, 9728), (8195, 4352), (8193, 5120), (8195, 5376), (8193, 6400), (4099, 17408)]


def rel_l2(got, want):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    return float(np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30))


@pytest.fixture
def backend(gpu):
    be = ops.Backend(0)
    yield be
    be.close()


def matvec(be, lin, x, rows, images=True):
    out = torch.full((1, rows), float("nan"), device=x.device)
    be.set_gemv_images(images)
    be.matvec_batch_k(out, lin, x, 1)
    be.set_gemv_images(True)
    return out.cpu().numpy()


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("tt", FORMATS)
def test_own_image_gemv(gpu, oracle, backend, tt, rows, cols):
    w = synth.make_weight(tt, rows, cols, seed=51, tag=tt)
    x = synth.make_act(cols, 1, seed=52, tag=cols)
    xd = torch.from_numpy(x).to(gpu)
    wd = torch.from_numpy(w).to(gpu)
    lin = backend.wrap_linear(tt, rows, cols, wd)
    plain = matvec(backend, lin, xd, rows, images=False)
    before = backend.mem_placed()
    got = matvec(backend, lin, xd, rows)
    assert backend.mem_placed() > before  # the image was built, so it was read
    # the same integers and the same float expression per 64 values, summed in
    # another order: 2^-24 a step over at most 272 of them
    assert rel_l2(got, plain) < 1e-6
    at = np.unique(np.r_[0:min(rows, 24), max(0, rows - 24):rows])
    wr = np.ascontiguousarray(w.reshape(rows, -1)[at])
    assert rel_l2(got[0, at], oracle.matvec(tt, wr, x)[0]) < 1e-5
    assert np.array_equal(got, matvec(backend, lin, xd, rows))


def test_q3_image_on_short_rows(gpu, oracle, backend):
    """Q3_K takes the image at widths where the others quantize in the launch,
    from 2560 (40 units)."""
    for tt, rows, cols, uses in ((po.TT_Q3_K, 3277, 2560, True), (po.TT_Q3_K, 3276, 2560, False),
                                 (po.TT_Q3_K, 3645, 2304, False), (po.TT_Q3_K, 32775, 256, False),
                                 (po.TT_Q2_K, 3277, 2560, False), (po.TT_Q5_K, 3277, 2560, False)):
        w = synth.make_weight(tt, rows, cols, seed=53, tag=rows)
        x = synth.make_act(cols, 1, seed=54, tag=1)
        xd = torch.from_numpy(x).to(gpu)
        wd = torch.from_numpy(w).to(gpu)
        lin = backend.wrap_linear(tt, rows, cols, wd)
        plain = matvec(backend, lin, xd, rows, images=False)
        before = backend.mem_placed()
        got = matvec(backend, lin, xd, rows)
        assert (backend.mem_placed() > before) == uses
        assert rel_l2(got, plain) < 1e-6


# 250 rows: the images' bytes are no multiple of the arena's alignment, so two
# adjacent weights' images are not adjacent, and the pair gets an image of its own
@pytest.mark.parametrize("rows", [256, 250])
@pytest.mark.parametrize("tt", FORMATS)
def test_own_image_pair_and_capture(gpu, oracle, backend, tt, rows):
    """Adjacent weights with adjacent images, in one launch; captured and
    replayed on new activations; and one weight of the pair alone."""
    cols = 5120
    w = synth.make_weight(tt, 2 * rows, cols, seed=55, tag=tt)
    wd = torch.from_numpy(w).to(gpu)
    half = wd.numel() // 2
    a = backend.wrap_linear(tt, rows, cols, wd.view(-1)[:half])
    b = backend.wrap_linear(tt, rows, cols, wd.view(-1)[half:])
    assert backend.lib.qhip_backend_alloc_scratch(backend._h, cols) == 0
    backend.set_mmq_images(False)  # the GEMV images alone
    before = backend.mem_placed()
    backend.prepare_linear(a)
    backend.prepare_linear(b)
    xd = torch.from_numpy(synth.make_act(cols, 1, seed=56, tag=0)).to(gpu)
    pair = torch.empty(2 * rows, device=gpu)
    placed = backend.mem_placed()
    row_bytes = {po.TT_Q2_K: 84, po.TT_Q3_K: 114, po.TT_Q5_K: 180}[tt] * (cols // 256)
    image = (row_bytes + 15) // 16 * 16 * rows
    adjacent = image % 256 == 0
    assert adjacent == (rows == 256)
    assert placed - before == 2 * ((image + 255) // 256 * 256)
    backend.matvec_pair(pair, a, b, xd[0])
    # in one launch from both images, or from one built for the pair
    assert backend.mem_placed() - placed == (0 if adjacent else (2 * image + 255) // 256 * 256)
    placed = backend.mem_placed()
    want = oracle.matvec(tt, w, xd.cpu().numpy())[0]
    assert rel_l2(pair.cpu().numpy(), want) < 1e-5
    second = matvec(backend, b, xd, rows)
    assert rel_l2(second[0], want[rows:]) < 1e-5
    assert np.array_equal(second[0], pair.cpu().numpy()[rows:])
    stream = torch.cuda.Stream()
    backend.set_stream(stream)
    out = torch.empty(1, rows, device=gpu)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        backend.matvec_batch_k(out, a, xd, 1)
    for tag in (1, 2, 3):
        x = synth.make_act(cols, 1, seed=56, tag=tag)
        xd.copy_(torch.from_numpy(x))
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy()[0], oracle.matvec(tt, w, x)[0][:rows]) < 1e-5
    assert backend.mem_placed() == placed  # the captured launch, too, read an image that was there


@pytest.mark.parametrize("tt", FORMATS)
def test_public_image_calls_keep_their_formats(gpu, tt):
    lib = _lib.load()
    assert lib.qhip_gemv_image_bytes(tt, 64, 5120) <= 0
    buf = torch.zeros(1 << 20, dtype=torch.uint8, device=gpu)
    assert lib.qhip_launch_gemv_prepare(tt, buf.data_ptr(), 64, 5120, buf.data_ptr(), None) != 0
