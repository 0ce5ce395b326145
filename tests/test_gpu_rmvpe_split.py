# -*- coding: utf-8 -*-
"""RMVPE's 2-D convolutions on split products: image heights from one deep row
up, across the wave counts of the tile rule, and values outside fp16's range."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from oracle import rmvpe_ref as R
from rvc_hip import synthetic as syn
from rvc_hip.rmvpe import HipRMVPE

pytestmark = pytest.mark.gpu

BLOCK = "unet.encoder.layers.%d.conv.1"


@pytest.fixture(scope="module")
def weights():
    return syn.make_rmvpe_weights(seed=6)


def _hidden(sd, x):
    m = HipRMVPE(sd)
    try:
        return m.mel2hidden_from_audio(x)[0]
    finally:
        m.close()


@pytest.mark.parametrize("frames", [4, 32, 33, 65, 97, 160])
def test_frame_counts(weights, frames):
    x = syn.make_rmvpe_audio(160 * (frames - 1) + 40, seed=frames)
    oracle = R.Rmvpe(weights)
    want = oracle.mel2hidden(oracle.mel(x)[None])[0]
    got = _hidden(weights, x)
    assert got.shape == want.shape
    # sums of up to 4608 products, then a recurrence and a sigmoid that damp them
    assert rel_l2(got, want) < 2e-6


@pytest.mark.parametrize("level", [0, 1, 4])
@pytest.mark.parametrize("exponent", [-60, -24, 24, 60])
def test_scale_of_the_values(weights, level, exponent):
    """ReLU passes a power of two through: the first conv of a block scaled up
    and the second down give the same block, up to rounding."""
    x = syn.make_rmvpe_audio(8000, seed=1)
    s = np.float32(2.0) ** exponent
    p = BLOCK % level
    sd = dict(weights)
    sd[p + ".conv.1.weight"] = sd[p + ".conv.1.weight"] * s
    sd[p + ".conv.1.bias"] = sd[p + ".conv.1.bias"] * s
    sd[p + ".conv.3.weight"] = sd[p + ".conv.3.weight"] / s
    assert rel_l2(_hidden(sd, x), _hidden(weights, x)) < 1e-6


def test_infinities(weights):
    """A channel of +inf under negative weights makes every sum -inf, which the
    ReLU turns into 0, as a bias far below the sums does."""
    x = syn.make_rmvpe_audio(8000, seed=2)
    p = BLOCK % 1
    inf, low = dict(weights), dict(weights)
    b = inf[p + ".conv.1.bias"].copy()
    b[3] = np.inf
    w = inf[p + ".conv.3.weight"].copy()
    w[:, 3] = -np.abs(w[:, 3]) - np.float32(1e-3)
    inf[p + ".conv.1.bias"], inf[p + ".conv.3.weight"] = b, w
    low[p + ".conv.4.bias"] = np.full_like(low[p + ".conv.4.bias"], -1e30)
    got, want = _hidden(inf, x), _hidden(low, x)
    assert np.isfinite(got).all()
    assert rel_l2(got, want) < 1e-6


@pytest.mark.parametrize("exponent", [16, 24])
def test_a_burst_takes_nothing_from_its_neighbours(weights, exponent):
    """A burst in silence, with the image's scale such that the burst is about
    2^20 times the silence, and the first encoder level cut down to one block:
    the frames that the burst does not reach share tiles with those it does, and
    are those of silence alone, within the error of two fp32 computations."""
    silence, F = np.zeros(16000, np.float32), 101
    burst = silence.copy()
    burst[8000:8800] = 0.5 * np.random.default_rng(1).standard_normal(800, dtype=np.float32)
    sd = dict(weights)
    p = "unet.encoder.bn."
    sd[p + "weight"] = np.full(1, 2.0 ** exponent, np.float32)
    sd[p + "bias"] = np.full(1, 2.0 ** (exponent - 18), np.float32)
    sd[p + "running_var"] = np.ones(1, np.float32)
    sd[p + "running_mean"] = np.full(1, np.log(1e-5), np.float32)
    for i in (1, 2, 3):
        for k in ("weight", "bias"):
            q = f"unet.encoder.layers.0.conv.{i}.conv.4.{k}"
            sd[q] = np.zeros_like(sd[q])
    m = HipRMVPE(sd)
    level = []
    for x in (silence, burst):
        m.mel2hidden_from_audio(x)
        level.append(m.read("cat0", (32, m.padded(F), 128))[16:])
    m.close()
    # the burst's samples lie in the windows of frames 47 .. 58, and each of the
    # block's two 3x3 convolutions reaches one frame further (the padding behind
    # frame 100 is as large as the burst)
    off = np.abs(level[1] - level[0]).max(axis=(0, 2)) / np.abs(level[0][:, :90]).max()
    assert (off[45:61] > 10).all()
    for near in (slice(40, 45), slice(61, 66)):
        assert rel_l2(level[1][:, near], level[0][:, near]) < 2e-6
