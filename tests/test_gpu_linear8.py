"""8-bit Linear products of more than 16 rows (routers, shared gates, small projections) against the
CPU restatement: the dense kernel's branches (scale groups of 128, a group shared by its two halves of
K, one half only, no biases, output and row remainders), and the sizes where the generic GEMM takes
over."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from mrun_amd import moe as M
from mrun_amd import synth
from oracle import oracle as O
from tests.helpers import beyond_rounding, stats

pytestmark = pytest.mark.gpu


def _weight(out, in_, group, biases=True):
    w = synth.normal_bf16(synth.seed(9, out + in_, synth.ROUTER_W), out * in_, 0.02).reshape(out, in_)
    q = synth.quantize(w, 8, group)
    return q if biases else dataclasses.replace(q, biases=None)


def _check(q, x, bias=None, rows=slice(None)):
    """R(x Wq^T) within accumulation-order rounding of the oracle's; with a bias, R(. + bias) of that,
    bit for bit (load.rs:302-305: its own rounding)."""
    dq = M.DeviceQTensor(q)
    got = M.bf16_bits(M.linear(M.bf16_tensor(x), dq))
    ref = O.linear(q, x[rows])
    assert beyond_rounding(got[rows], ref) == 0, stats(got[rows], ref)
    if bias is not None:
        want = synth.f32_to_bf16(synth.bf16_to_f32(got) + synth.bf16_to_f32(bias)[None, :])
        assert np.array_equal(M.bf16_bits(M.linear(M.bf16_tensor(x), dq, M.bf16_tensor(bias))), want)


# 384 inputs: three K steps per half, so that half a group of 128 lies in each; 320: five steps in one
@pytest.mark.parametrize("in_,group", [(384, 128), (2048, 128), (320, 64), (384, 64), (64, 64), (256, 32)])
@pytest.mark.parametrize("out", [1, 65, 512])
def test_dense_kernel_branches(in_, group, out):
    bias = synth.normal_bf16(synth.seed(9, 1, synth.ROUTER_BIAS), out, 0.1)
    for T in (17, 33, 70):
        x = synth.make_x(synth.Shape(in_, 1, 1, 32), T, config=9, layer=T)
        _check(_weight(out, in_, group), x, bias)
        _check(_weight(out, in_, group, biases=False), x)


@pytest.mark.parametrize("in_", [512, 4096])
@pytest.mark.parametrize("T", [16384, 16385])
def test_either_side_of_one_block_per_cu(in_, T):
    x = np.resize(synth.make_x(synth.Shape(in_, 1, 1, 32), 97, config=9, layer=1), (T, in_))
    _check(_weight(64, in_, 64), x, rows=np.r_[0:40, T - 40:T])
