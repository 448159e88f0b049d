"""GPU: the few-token MMQ from the fragment images of Q4_K, Q5_K and Q6_K that
keeps K inside the workgroup, through the Exec mirror: the edges of its element
groups (8 tokens), token tiles (32) and ranges, each wave count (four, eight and
twelve) at row counts that are no multiple of 32 and widths that leave waves
without a super-block, against the oracle; exact block integers of Q5_K; the
public fragment-image calls still refuse that format."""
import numpy as np
import pytest
import torch

import pyoracle as po
import qwen35_amd
from qwen35_amd import ops, synth
from test_gpu_mmq import rel_l2, to_dev, unit_scale_act, unit_scale_weight

TT = po.TT_Q5_K


def product(tt, wd, rows, cols, x, images=True):
    be = ops.Backend(0)
    be.set_mmq_images(images)
    lin = be.wrap_linear(tt, rows, cols, wd)
    out = torch.full((x.shape[0], rows), float("nan"), device=x.device)
    be.matvec_batch_k(out, lin, x, x.shape[0])
    placed = be.mem_placed()
    be.free_linear(lin)
    freed = placed - be.mem_placed()
    be.close()
    return out, freed


@pytest.mark.gpu
@pytest.mark.parametrize("tt", [po.TT_Q4_K, po.TT_Q5_K, po.TT_Q6_K])
@pytest.mark.parametrize("rows,cols", [(8195, 1024), (6570, 1280), (1000, 9216), (1640, 5120),
                                       (11000, 1280)])
def test_fragments_match_oracle(gpu, oracle, tt, rows, cols):
    w = synth.make_weight(tt, rows, cols, seed=61, tag=tt)
    wd = to_dev(w, gpu)
    pick = np.unique(np.r_[np.linspace(0, rows - 1, 40).astype(int), rows - 34:rows])
    for tokens in (2, 8, 9, 16, 17, 24, 25, 32, 33, 64, 65, 96, 97, 128, 129):
        x = synth.make_act(cols, tokens, seed=62, tag=tokens)
        tpick = np.unique(np.r_[np.linspace(0, tokens - 1, 12).astype(int), tokens - 1])
        xd = to_dev(x, gpu)
        got, image = product(tt, wd, rows, cols, xd)
        if tt == TT and tokens <= 128:
            assert image == (rows + 31) // 32 * 32 * (cols // 256) * 176
        # K is summed in the waves' order: a few f32 roundings of the sum, as the other MMQs
        want = oracle.matvec(tt, np.ascontiguousarray(w[pick]), np.ascontiguousarray(x[tpick]))
        assert rel_l2(got.cpu().numpy()[np.ix_(tpick, pick)], want) < 1e-5
        plain, image = product(tt, wd, rows, cols, xd, images=False)
        assert image == 0 and rel_l2(plain.cpu().numpy(), got.cpu().numpy()) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [7, 40])
def test_q5k_fragments_integers_exact(gpu, oracle, tokens):
    """d = dmin = 1 and activations of Q8_K scale 1, one super-block: every
    output is an exact integer below 2^24."""
    rows, cols = 32775, 256
    w = unit_scale_weight(TT, rows, cols, seed=63)
    x = unit_scale_act(cols, tokens, seed=64)
    pick = np.r_[0:64, rows - 40:rows]
    want = oracle.matvec(TT, np.ascontiguousarray(w[pick]), x)
    assert np.abs(want).max() < 2 ** 24 and np.array_equal(want, np.rint(want))
    got, image = product(TT, to_dev(w, gpu), rows, cols, to_dev(x, gpu))
    assert image > 0 and np.array_equal(got.cpu().numpy()[:, pick], want)


def test_public_fragment_calls_refuse_q5k():
    lib = qwen35_amd.load()
    assert lib.qhip_wd_image_bytes(TT, 64, 1024) == -1
    assert lib.qhip_launch_wd_prepare(TT, 16, 64, 1024, 16, 0) == 1  # hipErrorInvalidValue
