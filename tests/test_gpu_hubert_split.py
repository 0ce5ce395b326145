# -*- coding: utf-8 -*-
"""HuBERT's linear layers and stride-2 convs on split products: frame counts at
the edges of the tiles and of the tile rules, and values outside fp16's range."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from oracle import hubert_ref, nn_ref
from rvc_hip import synthetic as syn
from rvc_hip.hubert import HipHubert

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def weights():
    return syn.make_hubert_weights(syn.HUBERT_BASE, seed=6)


@pytest.fixture(scope="module")
def hub(weights):
    return HipHubert(weights)


@pytest.mark.parametrize("L", [1, 31, 32, 33, 65, 129, 226, 400])
def test_frame_counts(weights, hub, L):
    T = 400 + 320 * (L - 1)
    x = syn.make_hubert_input(T, seed=L)
    with nn_ref.conv_formulation("taps"):
        want = hubert_ref.HubertRef(weights).encode(x)
    got = hub.encode(x)
    assert got.shape == want.shape == (1, L, 768)
    # 12 layers, sums of 768 and 3072 products: about 1e-6 on either side
    assert rel_l2(got, want) < 5e-6


@pytest.mark.parametrize("exponent", [-60, -20, 20, 60])
def test_scale_of_the_values(weights, hub, exponent):
    """The projection is linear: its input (the affine of the LayerNorm in
    front) and bias scaled by a power of two scale its output, up to rounding."""
    s = np.float32(2.0) ** exponent
    scaled = {k: v * s if k.startswith("feature_projection.layer_norm") or k == "feature_projection.projection.bias"
              else v for k, v in weights.items()}
    other = HipHubert(scaled)
    x = syn.make_hubert_input(12000, seed=2)
    L = hub.frames(12000)
    hub.encode(x)
    other.encode(x)
    assert rel_l2(other.read("proj", (1, 768, L)) / s, hub.read("proj", (1, 768, L))) < 1e-6
    other.close()


def _other_width(hidden, ffn, L):
    """rel L2 of a two-layer model of another width against the oracle."""
    sd = syn.make_hubert_weights(syn.HubertGeometry(conv_dim=64, hidden=hidden, n_layers=2, ffn=ffn), seed=hidden)
    x = syn.make_hubert_input(400 + 320 * (L - 1), seed=L)
    with nn_ref.conv_formulation("taps"):
        want = hubert_ref.HubertRef(sd).encode(x)
    m = HipHubert(sd)
    got = m.encode(x)
    m.close()
    assert got.shape == want.shape == (1, L, hidden)
    return rel_l2(got, want)


@pytest.mark.parametrize("hidden,ffn,L", [(1152, 4608, 129), (1536, 6144, 129)])
def test_more_than_1024_channels(hidden, ffn, L):
    """36 and 48 tiles of LayerNorm statistics, at a frame count at which q/k/v
    and the FFN run on 64-row tiles of four waves."""
    # sums of up to 6144 products, as above
    assert _other_width(hidden, ffn, L) < 5e-6


@pytest.mark.parametrize("hidden,ffn,L", [(384, 1536, 33), (384, 1536, 460), (576, 2304, 40), (576, 2304, 300),
                                          (960, 3840, 40), (960, 3840, 170), (1344, 5376, 97)])
def test_uneven_shares_of_the_waves(hidden, ffn, L):
    """Widths whose 16-channel steps do not divide evenly among the four or
    eight waves of a tile, with the LayerNorm applied on the way in."""
    assert _other_width(hidden, ffn, L) < 5e-6


@pytest.mark.parametrize("hidden,ffn,L", [(192, 768, 40), (288, 3072, 40), (288, 3072, 300), (480, 1920, 70),
                                          (384, 1500, 40)])
def test_widths_the_split_products_do_not_take(hidden, ffn, L):
    """At most 256 channels, or not a multiple of 64: the fp32 GEMMs, among them
    the 3072-channel reduction in two splits with its reduce launch, and the
    LayerNorms as launches of their own."""
    assert _other_width(hidden, ffn, L) < 5e-6


def test_a_click_takes_nothing_from_its_neighbours(weights):
    """Two opposite clicks of 1e6 in noise of 1e-3, no GroupNorm bias: the frames
    beside them share tiles of the first stride-2 conv with theirs, 2^27 times as
    large.  What the normalisation leaves of the noise is off by about 1e-3 on
    either side (its rounding), beside the clicks as elsewhere."""
    sd = dict(weights)
    key = "feature_extractor.conv_layers.0.layer_norm.bias"
    sd[key] = np.zeros_like(sd[key])
    x = 1e-3 * np.random.default_rng(1).standard_normal((1, 34000), dtype=np.float32)
    x[0, 16000], x[0, 16400] = 1e6, -1e6
    with nn_ref.conv_formulation("taps"):
        want = hubert_ref.HubertRef(sd).feature_extractor(x)[0]  # [106][512]
    m = HipHubert(sd)
    m.encode(x)
    got = m.read("feats", (512, 106)).T
    m.close()
    off = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    beside = np.r_[off[44:49], off[52:57]]
    assert (off[49:52] < 5e-6).all()
    assert beside.max() < 1.6 * np.median(off)
