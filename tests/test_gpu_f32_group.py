"""f32 blocks on the grouped kernel (weights kept in registers for a tile of rows): input widths at
the edges of its three instantiations, batches on either side of the sort by expert (36 million pairs
times weights of a projection, and logits too small to hold the routing), tiles of 8 to 64 rows and
more, and rows independent of all of these."""
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
    synth.Shape(hidden=256, experts=64, top_k=4, intermediate=128, shared=128),  # never sorted at these sizes
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


# sorted from the batch after the first size given: tiles of 8 rows, then of 16 and more
@pytest.mark.parametrize("shape,Ts", [
    (synth.Shape(hidden=1024, experts=8, top_k=2, intermediate=1024, shared=1024), (17, 18, 75, 600)),
    (synth.Shape(hidden=512, experts=40, top_k=4, intermediate=512, shared=0), (34, 35, 300, 2100)),
    (synth.Shape(hidden=2048, experts=8, top_k=1, intermediate=512, shared=512), (34, 35, 200, 4100)),
])
def test_rows_do_not_depend_on_the_tiles(shape, Ts):
    fb = synth.make_block_f32(shape, config=30)
    dev = M.SparseMoeF32(fb)
    x = np.resize(synth.make_x_f32(shape, 75, config=30), (max(Ts), shape.hidden))
    check(fb, dev, x[:Ts[1]], f"{shape.name} T={Ts[1]}")
    one = dev.forward(f32_dev(x[:Ts[0]])).cpu().numpy().view(np.uint32)
    for T in Ts[1:]:
        got = dev.forward(f32_dev(x[:T])).cpu().numpy().view(np.uint32)
        assert np.array_equal(got[:Ts[0]], one), T
        assert np.array_equal(got, np.resize(got[:75], got.shape)), T


def test_every_row_on_one_expert():
    """A router that sends every token to the same expert: its rows are cut into tiles like any."""
    shape = synth.Shape(hidden=512, experts=16, top_k=1, intermediate=512, shared=0)
    fb = synth.make_block_f32(shape, config=31)
    fb.router[:] = 0.0  # equal logits: the lowest id
    dev = M.SparseMoeF32(fb)
    x = synth.make_x_f32(shape, 300, config=31)
    got = check(fb, dev, x, "one expert T=300").view(np.uint32)
    part = dev.forward(f32_dev(x[:9])).cpu().numpy().view(np.uint32)
    assert np.array_equal(part, got[:9])


def test_more_tiles_than_a_grid_holds():
    """400,000 rows of 16 pairs are 100,000 tiles of 64 and 50,000 pieces of plain rows: larger tiles."""
    shape = synth.Shape(hidden=32, experts=32, top_k=16, intermediate=32, shared=32)
    dev = M.SparseMoeF32(synth.make_block_f32(shape, config=32))
    x = f32_dev(synth.make_x_f32(shape, 1000, config=32)).repeat(400, 1)
    full = dev.forward(x)
    part = dev.forward(x[:1000].contiguous())
    assert torch.equal(full.view(400, 1000, 32), part.expand(400, -1, -1))
