"""Prefill batches of the checkpoint formats the grouped GEMM of moe_fmt.hip runs (4-bit groups of
32 and 128, 8-bit groups of 32, 64 and 128, bf16 weights), against the CPU restatement, with the
bars of test_gpu_parity.py: at the edges of its 32- and 64-row tiles, with and without a shared
expert, without biases, with gate/up and down in different formats, and rows independent of the
batch's tile size."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from mrun_amd import moe as M
from mrun_amd import synth
from oracle import oracle as O
from tests.helpers import assert_close
from tests.test_gpu_parity import _without_biases, run_block

pytestmark = pytest.mark.gpu

BASE = synth.Shape(hidden=1024, experts=8, top_k=2, intermediate=512, shared=512)
FORMATS = [(4, 32), (4, 128), (8, 32), (8, 64), (8, 128), (16, 64)]


def _host(bits, group, layer=0, **kw):
    shape = dataclasses.replace(BASE, group=group, **kw)
    return synth.make_block(shape, config=synth.CFG_PLUMBING, layer=layer, expert_bits=bits)


def _x(shape, T, layer=0):
    return synth.make_x(shape, T, config=synth.CFG_PLUMBING, layer=layer)


# 33 and 97 rows: 32-row tiles (experts average at most 28 rows); 130 and 300: 64-row tiles
@pytest.mark.parametrize("T", [33, 97, 130, 300])
@pytest.mark.parametrize("bits,group", FORMATS)
def test_format_matches_oracle(bits, group, T):
    hb = _host(bits, group, layer=group)
    run_block(hb, M.SparseMoe(hb), _x(hb.shape, T, T), f"{bits}-bit group {group} T={T}")


@pytest.mark.parametrize("bits,group", FORMATS)
def test_rows_keep_their_bits_across_tile_sizes(bits, group):
    """A row's result is the same on 64-row tiles (T = 300) and 32-row ones (T = 97)."""
    hb = _host(bits, group, layer=7)
    dev = M.SparseMoe(hb)
    x = _x(hb.shape, 300)
    full = M.bf16_bits(dev.forward(M.bf16_tensor(x)))
    part = M.bf16_bits(dev.forward(M.bf16_tensor(x[:97])))
    assert np.array_equal(part, full[:97])


@pytest.mark.parametrize("kw", [dict(shared=0), dict(shared=1024), dict(top_k=1), dict(hidden=1536)])
@pytest.mark.parametrize("bits,group", [(4, 32), (8, 64), (16, 64)])
def test_block_variants(bits, group, kw):
    """No shared expert; one of another width (generic GEMMs); one expert per token (no room for
    sums of 32 inputs in the workspace: generic GEMMs); hidden 3 x 512."""
    hb = _host(bits, group, **kw)
    run_block(hb, M.SparseMoe(hb), _x(hb.shape, 130), f"{bits}-bit group {group} {kw}")


@pytest.mark.parametrize("bits,group", [f for f in FORMATS if f[0] != 16])
def test_without_biases(bits, group):
    hb = _without_biases(_host(bits, group, layer=3))
    for T in (40, 130):
        run_block(hb, M.SparseMoe(hb), _x(hb.shape, T), f"{bits}-bit group {group} no biases T={T}")


@pytest.mark.parametrize("gate,down", [((4, 64), (8, 64)), ((8, 64), (4, 64)), ((4, 64), (4, 32)),
                                       ((4, 32), (8, 64)), ((8, 128), (4, 32)), ((4, 64), (16, 64)),
                                       ((16, 64), (8, 64))])
def test_mixed_formats(gate, down):
    """Gate/up and down in different formats (mixed-precision conversions), on the grouped GEMMs
    where the sums one product writes are those the next one reads, else on the generic ones."""
    hb, other = _host(*gate, layer=4), _host(*down, layer=5)
    hb.down_proj, hb.sh_down_proj = other.down_proj, other.sh_down_proj
    for T in (40, 300):
        run_block(hb, M.SparseMoe(hb), _x(hb.shape, T), f"gate/up {gate} down {down} T={T}")


# 128 experts: enough work for the grouped GEMM (groups of 32 and bf16 weights: the generic one); with
# 8, only group 64 takes it; 640 inputs: the generic one
@pytest.mark.parametrize("hidden,experts", [(1024, 128), (1024, 8), (640, 8)])
@pytest.mark.parametrize("bits,group", [(4, 64)] + FORMATS)
def test_gather_qmm(bits, group, hidden, experts):
    """gather_qmm above 16 indices in every format: unsorted indices, x rows shared by two."""
    q = _host(bits, group, layer=6, hidden=hidden, experts=experts).gate_proj
    n, rows = 150, 75
    ids = np.random.default_rng(1).integers(0, q.experts, n).astype(np.uint32)
    x = _x(synth.Shape(q.in_, 1, 1, 32), rows)
    got = M.bf16_bits(M.gather_qmm(M.bf16_tensor(x), M.DeviceQTensor(q), M.u32_tensor(ids)))
    ref = O.gather_qmm(q, x, ids)
    assert_close(got, ref, what=f"gather_qmm {bits}-bit group {group} in {hidden} experts {experts}")


@pytest.mark.parametrize("T", [900, 1500, 2600, 6000])
@pytest.mark.parametrize("bits,group", [(4, 32), (8, 64), (16, 64)])
def test_rows_keep_their_bits_across_item_rounds(bits, group, T):
    """Workgroups that take one to six items each, split evenly over fewer workgroups or not: every
    row as in a batch of one item per workgroup."""
    hb = _host(bits, group, layer=8, intermediate=1024, shared=1024)
    dev = M.SparseMoe(hb)
    x = np.resize(_x(hb.shape, 97), (T, hb.shape.hidden))
    full = M.bf16_bits(dev.forward(M.bf16_tensor(x)))
    part = M.bf16_bits(dev.forward(M.bf16_tensor(x[:97])))
    assert np.array_equal(full, np.resize(part, full.shape))


# 6,000 rows of 8 experts: three rounds of 64-row tiles per workgroup; 400 rows of 128 experts (25
# rows each): more 32-row tiles than workgroups
@pytest.mark.parametrize("T,kw", [(6000, {}), (400, dict(hidden=512, experts=128, top_k=8))])
@pytest.mark.parametrize("bits,group", [(4, 64)] + FORMATS)
def test_a_non_finite_row_stays_alone(bits, group, T, kw):
    """A token row of infinities or NaN (an uninitialised padding row) changes no other row: nothing
    of one tile's products reaches the next tile of the same workgroup."""
    hb = _host(bits, group, layer=9, **kw)
    dev = M.SparseMoe(hb)
    x = np.resize(_x(hb.shape, 97), (T, hb.shape.hidden))
    clean = M.bf16_bits(dev.forward(M.bf16_tensor(x)))
    bad = np.array([3, T // 2, T - 5])
    x[bad] = np.array([0x7F80, 0xFF80, 0x7FC0], dtype=np.uint16)[:, None]  # inf, -inf, NaN
    got = M.bf16_bits(dev.forward(M.bf16_tensor(x)))
    others = np.setdiff1d(np.arange(T), bad)
    wrong = others[np.any(got[others] != clean[others], axis=1)]
    assert wrong.size == 0, f"{wrong.size} other rows changed, the first {wrong[:4]}"
