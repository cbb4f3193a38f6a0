"""f32 blocks on the grouped kernel (weights kept in registers for every row that meets them): input
widths at the edges of its three instantiations, batches on either side of the sort by expert (a
third of a pair per expert, and logits too small to hold the routing), and rows independent of both."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from mrun_amd import moe as M
from mrun_amd import synth
from tests.test_gpu_f32 import check, f32_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter", [(32, 2048), (512, 544), (1024, 512), (1056, 96), (2048, 1024),
                                          (2080, 64)])  # 2080: above the grouped kernel's widths
def test_input_widths(hidden, inter):
    shape = synth.Shape(hidden=hidden, experts=12, top_k=3, intermediate=inter, shared=inter)
    fb = synth.make_block_f32(shape, config=27)
    dev = M.SparseMoeF32(fb)
    for T in (1, 9, 70):
        check(fb, dev, synth.make_x_f32(shape, T, config=27, layer=T), f"{shape.name} T={T}")


@pytest.mark.parametrize("shape", [
    synth.Shape(hidden=256, experts=64, top_k=4, intermediate=128, shared=128),  # sorted from T = 6
    synth.Shape(hidden=256, experts=8, top_k=8, intermediate=128),               # logits too small
    synth.Shape(hidden=256, experts=32, top_k=2, intermediate=128, shared=64),   # another shared width
])
def test_rows_do_not_depend_on_the_grouping(shape):
    fb = synth.make_block_f32(shape, config=28)
    dev = M.SparseMoeF32(fb)
    x = synth.make_x_f32(shape, 75, config=28)
    full = dev.forward(f32_dev(x)).cpu().numpy().view(np.uint32)
    for T in (1, 7, 8, 9, 64):
        part = dev.forward(f32_dev(x[:T])).cpu().numpy().view(np.uint32)
        assert np.array_equal(part, full[:T]), T
    check(fb, dev, x, shape.name)


def test_more_row_pieces_than_a_grid_holds():
    """530,000 rows are 66,250 pieces: the per-row kernel runs them, with the same bits."""
    shape = synth.Shape(hidden=32, experts=4, top_k=1, intermediate=32, shared=32)
    dev = M.SparseMoeF32(synth.make_block_f32(shape, config=29))
    x = f32_dev(synth.make_x_f32(shape, 1000, config=29)).repeat(530, 1)
    full = dev.forward(x)
    part = dev.forward(x[:1000].contiguous())
    assert torch.equal(full.view(530, 1000, 32), part.expand(530, -1, -1))
