"""GPU: the prompt MMQ from plane and activation images, through the Exec
mirror: every format and every switch of its dispatch (the token count it
starts at, 64- against 128-token tiles, sliced and whole tiles) at row counts
that are no multiple of a tile, against the oracle; exact block integers at
unit scales and at the largest scales and values; the activation image byte
for byte; a captured launch replayed; the activation memo across families."""
import ctypes

import numpy as np
import pytest
import torch

import pyoracle as po
from qwen35_amd import _lib, ops, synth
from test_gpu_mmq import rel_l2, to_dev, unit_scale_act, unit_scale_weight

pytestmark = pytest.mark.gpu
TOL = 1e-5
FORMATS = [po.TT_Q6_K, po.TT_Q5_K, po.TT_Q2_K, po.TT_Q3_K, po.TT_IQ4_XS, po.TT_IQ3_XXS, po.TT_IQ3_S]
START = 129  # the token count the route starts at on a small weight (Q6_K reads the plane image from 65)


@pytest.fixture
def backend(gpu):
    be = ops.Backend(0)
    yield be
    be.close()


def product(be, tt, wd, rows, cols, x, images=True):
    tokens = x.shape[0]
    lin = be.wrap_linear(tt, rows, cols, wd)
    be.set_mmq_images(images)
    out = torch.full((tokens, rows), float("nan"), device=x.device)
    be.matvec_batch_k(out, lin, x, tokens)
    be.set_mmq_images(True)
    placed = be.mem_placed()
    be.free_linear(lin)
    return out, placed - be.mem_placed()


@pytest.mark.parametrize("tt", FORMATS)
def test_planes_match_oracle(gpu, oracle, backend, tt):
    rows, cols = 333, 2048
    w = synth.make_weight(tt, rows, cols, seed=41, tag=tt)
    wd = to_dev(w, gpu)
    for tokens in (64, 65, START - 1, START, 130, 256, 257, 300):
        x = synth.make_act(cols, tokens, seed=42, tag=tokens)
        xd = to_dev(x, gpu)
        got, image = product(backend, tt, wd, rows, cols, xd)
        assert rel_l2(got.cpu().numpy(), oracle.matvec(tt, w, x)) < TOL
        assert (image > 0) == (tokens >= (65 if tt == po.TT_Q6_K else START))
        again, _ = product(backend, tt, wd, rows, cols, xd)
        assert torch.equal(got, again)  # the slices are added in a fixed order
        plain, image = product(backend, tt, wd, rows, cols, xd, images=False)
        assert image == 0 and rel_l2(plain.cpu().numpy(), got.cpu().numpy()) < 1e-6


# 17408 x 256 rows and K of one super-block: more than a round of whole tiles and
# nothing to slice; 66 x 8192: a few tiles, sliced; 4224 x 2048: a full round of
# 128-token tiles of 256 rows and a sliced remainder; 700 x 1024 and x 2304: 18
# whole tiles and 36 pieces of sliced ones, no multiples of the eight XCDs
@pytest.mark.parametrize("tt", [po.TT_Q6_K, po.TT_Q3_K, po.TT_Q5_K])
@pytest.mark.parametrize("rows,cols,tokens", [(17408, 256, 250), (66, 8192, 257), (4224, 2048, 2100),
                                              (700, 1024, 150), (700, 2304, 150)])
def test_planes_grids(gpu, oracle, backend, tt, rows, cols, tokens):
    w = synth.make_weight(tt, rows, cols, seed=43, tag=tt)
    x = synth.make_act(cols, tokens, seed=44)
    wd, xd = to_dev(w, gpu), to_dev(x, gpu)
    got, _ = product(backend, tt, wd, rows, cols, xd)
    pick = np.unique(np.linspace(0, rows - 1, 70).astype(int))
    tpick = np.unique(np.linspace(0, tokens - 1, 60).astype(int))
    want = oracle.matvec(tt, np.ascontiguousarray(w[pick]), np.ascontiguousarray(x[tpick]))
    assert rel_l2(got.cpu().numpy()[np.ix_(tpick, pick)], want) < TOL
    plain, _ = product(backend, tt, wd, rows, cols, xd, images=False)
    assert rel_l2(plain.cpu().numpy(), got.cpu().numpy()) < 1e-6


@pytest.mark.parametrize("tt", [po.TT_Q6_K, po.TT_Q5_K, po.TT_Q3_K, po.TT_Q2_K, po.TT_IQ4_XS])
@pytest.mark.parametrize("tokens", [140, 270])
def test_planes_integers_exact(gpu, oracle, backend, tt, tokens):
    """d = dmin = 1 in one super-block of a row and 0 in the others, activations
    of Q8_K scale 1: every output is that block's exact integer (below 2^24)."""
    rows, cols = 70, 2048
    w = unit_scale_weight(tt, rows, cols, seed=45)
    blk = w.reshape(rows, 8, -1)
    at = {po.TT_Q6_K: 208, po.TT_Q3_K: 108, po.TT_Q2_K: 80}.get(tt, 0)
    blk[:, np.arange(8) != 5, at:at + (4 if tt in (po.TT_Q5_K, po.TT_Q2_K) else 2)] = 0
    x = unit_scale_act(cols, tokens, seed=46)
    want = oracle.matvec(tt, w, x)
    assert np.abs(want).max() < 2 ** 24 and np.array_equal(want, np.rint(want))
    got, image = product(backend, tt, to_dev(w, gpu), rows, cols, to_dev(x, gpu))
    assert image > 0 and np.array_equal(got.cpu().numpy(), want)


def test_planes_largest_values(gpu, oracle, backend):
    """Q3_K's product -32 x -4 = 128 (held as -128) and Q6_K's -128 x -32 =
    4096 in every place, activations +-127: the ends of the planes' range."""
    cols, rows, tokens = 256, 64, 140
    x = np.where(np.arange(cols) % 3 == 0, -127.0, 127.0).astype(np.float32)[None].repeat(tokens, 0)
    w3 = np.zeros((rows, 110), np.uint8)  # scales 0 (-32), q2 0 and hmask 0 (-4)
    w3[:, 108:110] = np.array([1.0], np.float16).view(np.uint8)
    w6 = np.zeros((rows, 210), np.uint8)  # ql, qh 0 (-32)
    w6[:, 192:208] = 0x80
    w6[:, 208:210] = np.array([1.0], np.float16).view(np.uint8)
    for tt, w in ((po.TT_Q3_K, w3), (po.TT_Q6_K, w6)):
        got, image = product(backend, tt, to_dev(w, gpu), rows, cols, to_dev(x, gpu))
        assert image > 0 and np.array_equal(got.cpu().numpy(), oracle.matvec(tt, w, x))


@pytest.mark.parametrize("shift", [0, 1])  # x 16-byte aligned, and 4 bytes past it
def test_activation_image_bytes(gpu, oracle, shift):
    """The image holds the Q8_K rows' bytes: quants 512 v + 16 t, sums as f16,
    scales; tokens past the end are zeros."""
    cols, tokens = 768, 45
    x = synth.make_act(cols, tokens, seed=47)
    x[3, 300] = np.nan
    x[5, :256] = 0.0
    buf = torch.empty(tokens * cols + 4, device=gpu)
    xd = buf[shift:shift + tokens * cols].view(tokens, cols)
    xd.copy_(to_dev(x, gpu))
    dll = ctypes.CDLL(str(_lib.LIB_PATH))
    quantize = dll["_ZN4qhip23launch_quantize_mmq_actEPKfPviiP12ihipStream_t"]
    quantize.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    out = torch.empty(2 * 3 * 9344, dtype=torch.uint8, device=gpu)
    assert quantize(xd.data_ptr(), out.data_ptr(), cols, tokens, torch.cuda.current_stream().cuda_stream) == 0
    img = out.cpu().numpy().reshape(2, 3, 9344)
    act = oracle.quantize_act(po.TT_Q6_K, x).reshape(tokens, 3, 292)
    for tg in range(2):
        n = min(32, tokens - 32 * tg)
        a = act[32 * tg:32 * tg + n].transpose(1, 0, 2)  # [sb, token, byte]
        q = img[tg, :, :8192].reshape(3, 16, 32, 16).transpose(0, 2, 1, 3).reshape(3, 32, 256)
        assert np.array_equal(q[:, :n], a[:, :, 4:260]) and not q[:, n:].any()
        s = img[tg, :, 8192:9216].copy().view(np.float16).reshape(3, 2, 4, 16, 4).transpose(0, 1, 3, 2, 4).reshape(3, 32, 16)
        assert np.array_equal(s[:, :n], np.ascontiguousarray(a[:, :, 260:]).view(np.int16).astype(np.float16))
        d = img[tg, :, 9216:].copy().view(np.float32)
        assert np.array_equal(d[:, :n], np.ascontiguousarray(a[:, :, :4]).view(np.float32)[..., 0])


def test_planes_captured_and_memo(gpu, oracle, backend):
    """A captured launch replays on new activations; with the memo on, a second
    product of the same x reuses the image, and a product of another activation
    family does not meet it."""
    tt, rows, cols, tokens = po.TT_Q5_K, 300, 1024, 150
    w = synth.make_weight(tt, rows, cols, seed=48)
    wd = to_dev(w, gpu)
    lin = backend.wrap_linear(tt, rows, cols, wd)
    assert backend.prepare_linear(lin) == 0
    xs = [synth.make_act(cols, tokens, seed=49 + i) for i in range(3)]
    x, out = to_dev(xs[0], gpu), torch.empty((tokens, rows), device=gpu)
    side = torch.cuda.Stream()
    backend.set_stream(side)
    with torch.cuda.stream(side):
        backend.matvec_batch_k(out, lin, x, tokens)  # scratch and workspace grow here
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        backend.matvec_batch_k(out, lin, x, tokens)
    for xi in xs:
        x.copy_(to_dev(xi, gpu))
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy(), oracle.matvec(tt, w, xi)) < TOL
    backend.set_stream(torch.cuda.current_stream())
    backend.set_act_memo(True)
    h0, m0 = backend.act_stats()
    first, second, few = (torch.empty((tokens, rows), device=gpu) for _ in range(3))
    backend.matvec_batch_k(first, lin, x, tokens)
    backend.matvec_batch_k(second, lin, x, tokens)
    backend.set_mmq_images(False)  # another weight without an image: its GGUF rows, on Q8_K rows
    other = wd.clone()
    backend.matvec_batch_k(few, backend.wrap_linear(tt, rows, cols, other), x, tokens)
    backend.set_mmq_images(True)
    assert torch.equal(first, second) and rel_l2(few.cpu().numpy(), first.cpu().numpy()) < 1e-6
    h1, m1 = backend.act_stats()
    assert (h1 - h0, m1 - m0) == (1, 2)


@pytest.mark.parametrize("tt", [po.TT_Q3_K, po.TT_Q6_K])
@pytest.mark.parametrize("room", [True, False])
def test_planes_captured_after_reservation(gpu, oracle, backend, tt, room):
    """alloc_scratch_k and prepare_linear make a prompt capturable without an
    eager run before it, also at a token count that is no whole group of 32;
    where the budget holds only the Q8_K rows, the product runs on those (Q6_K
    from the plane image still)."""
    rows, cols, tokens = 300, 1024, 133
    w = synth.make_weight(tt, rows, cols, seed=51)
    wd = to_dev(w, gpu)
    lin = backend.wrap_linear(tt, rows, cols, wd)
    assert backend.prepare_linear(lin) == 0
    placed = backend.mem_placed()
    if not room:
        backend.set_mem_budget(placed + cols // 256 * 292 * tokens + 256)
    assert backend.lib.qhip_backend_alloc_scratch_k(backend._h, cols, tokens) == 0
    assert (backend.mem_placed() - placed >= cols // 256 * 292 * 160) == room
    x, out = torch.empty((tokens, cols), device=gpu), torch.empty((tokens, rows), device=gpu)
    side = torch.cuda.Stream()
    backend.set_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        backend.matvec_batch_k(out, lin, x, tokens)
    for i in range(3):
        xi = synth.make_act(cols, tokens, seed=52 + i)
        x.copy_(to_dev(xi, gpu))
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy(), oracle.matvec(tt, w, xi)) < TOL
    backend.set_stream(torch.cuda.current_stream())
    if tt == po.TT_Q6_K and not room:  # the bits of the public image product, unsplit as under the capture
        rows_out = ops.mul_mat_image(tt, ops.mmq_image(tt, wd, rows, cols), ops.quantize_act(tt, x), rows, cols, tokens)
        assert torch.equal(rows_out, out)


def image_bytes(tt, rows, cols, planes):
    group = {po.TT_Q6_K: (16512, 6720), po.TT_Q5_K: (17664, 5632), po.TT_Q3_K: (8320, 0), po.TT_Q2_K: (9472, 0),
             po.TT_IQ4_XS: (16512, 0)}[tt]  # per 32 rows and 256 values: planes, fragments
    return (rows + 31) // 32 * (cols // 256) * group[0 if planes else 1]


# both sides of each line of the dispatch: tokens -> plane image, fragment image
# or neither
@pytest.mark.parametrize("tt,rows,cols,routes", [
    (po.TT_Q6_K, 1640, 5120, {96: "frag", 97: "planes"}),
    (po.TT_Q6_K, 2720, 8448, {96: "frag"}), (po.TT_Q6_K, 2752, 8448, {64: "frag", 65: "planes"}),
    (po.TT_Q6_K, 16384, 1024, {65: "planes"}), (po.TT_Q6_K, 16640, 4096, {96: "frag", 97: "planes"}),
    (po.TT_Q6_K, 20512, 2048, {65: "planes"}), (po.TT_Q6_K, 14336, 3072, {64: "frag", 65: "planes"}),
    (po.TT_Q5_K, 1640, 5120, {128: "frag", 129: "planes"}),
    # the tile MMQ in one full round | rows of few super-blocks in many rows
    (po.TT_Q5_K, 16384, 1024, {96: "frag", 97: None, 128: None, 129: "planes"}),
    (po.TT_Q5_K, 20512, 1024, {96: "frag", 97: "planes"}),
    (po.TT_Q2_K, 2458, 5120, {64: None, 65: "planes"}), (po.TT_Q2_K, 2457, 5120, {128: None, 129: "planes"}),
    (po.TT_Q3_K, 1639, 5120, {64: None, 65: "planes"}), (po.TT_Q3_K, 1638, 5120, {128: None, 129: "planes"}),
    (po.TT_Q3_K, 3482, 5120, {24: None, 25: "planes"}), (po.TT_Q3_K, 3481, 5120, {64: None, 65: "planes"}),
    # fewer than eight super-blocks a row: from 9/16 of a tile per CU, of 512 values two
    (po.TT_IQ4_XS, 4096, 1024, {256: None, 257: "planes"}), (po.TT_IQ4_XS, 8192, 512, {448: None, 449: "planes"}),
    # three token tiles of long rows: up to 9/8 tiles per CU, and past 3/2
    (po.TT_IQ4_XS, 12288, 4096, {192: "planes"}), (po.TT_IQ4_XS, 12416, 4096, {128: None, 192: None, 193: "planes"}),
])
def test_prompt_routes(gpu, oracle, backend, tt, rows, cols, routes):
    w = synth.make_weight(tt, rows, cols, seed=55, tag=rows).reshape(rows, -1)
    wd = to_dev(w, gpu)
    at = np.unique(np.r_[np.linspace(0, rows - 1, 40).astype(int), rows - 3:rows])
    for tokens, route in routes.items():
        x = synth.make_act(cols, tokens, seed=56)
        got, image = product(backend, tt, wd, rows, cols, to_dev(x, gpu))
        assert rel_l2(got.cpu().numpy()[:, at], oracle.matvec(tt, np.ascontiguousarray(w[at]), x)) < TOL
        assert image == (0 if route is None else image_bytes(tt, rows, cols, route == "planes")), tokens
