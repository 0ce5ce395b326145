# -*- coding: utf-8 -*-
"""The decoder's ResBlocks on split products (conv_split.hip,
resblock_pair.hip): chunk lengths at the edges of the kernels' tiles, values
outside fp16's range, and sums that hold an infinity."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from oracle import nn_ref, vits_ref
from rvc_hip import synthetic as syn
from rvc_hip.synth import HipSynthesizer

pytestmark = pytest.mark.gpu


def _geom(upsample_initial, n_ups):
    return syn.Geometry(phone_dim=64, hidden=48, filter_channels=96, n_layers=1, gin=32, n_spk=2,
                        upsample_initial=upsample_initial, upsample_rates=(2,) * n_ups,
                        upsample_kernels=(4,) * n_ups, sr=100 * 2 ** n_ups)


# stage channels 128 / 64 / 32 (the fused groups) and 192 / 96 (a launch per conv)
GEOMS = {"fused": _geom(256, 3), "plain": _geom(384, 2)}


@pytest.fixture(scope="module")
def decoders():
    out = {}
    for name, geom in GEOMS.items():
        w = syn.make_weights(geom, seed=4)
        out[name] = (geom, w, HipSynthesizer(w, sr=geom.sr), vits_ref.GeneratorNSF(w, vits_ref.VitsConfig(w, sr=geom.sr)))
    return out


@pytest.mark.parametrize("name,P", [("fused", P) for P in (1, 2, 15, 16, 17, 33, 64, 127, 129, 2100, 8300)] +
                         [("plain", P) for P in (1, 17, 32, 33, 129, 1601, 3001)])
def test_tile_edges(decoders, name, P):
    geom, _, hip, ref = decoders[name]
    d = syn.make_dec_inputs(geom, P, seed=P)
    with nn_ref.conv_formulation("taps"):
        want = ref.forward(d["z"], d["f0"], d["g"], d["ns"])
    got = hip.dec.forward(d["z"], d["f0"], d["g"], d["ns"])
    # 18 convs deep, sums of up to 192 * 11 products: 2^-24 sqrt(2112) per
    # conv, added in quadrature, below 1e-5 on both sides
    assert rel_l2(got, want) < 2e-5
    assert np.abs(got - want).max() < 1e-4


@pytest.mark.parametrize("name", sorted(GEOMS))
@pytest.mark.parametrize("exponent", [-60, -24, -7, 12, 24, 60])
def test_scale_of_the_values(decoders, name, exponent):
    """Leaky ReLU and the convolutions are homogeneous: with every source of
    the decoder (conv_pre, cond, noise convs, biases) scaled by a power of two
    each stage is the unscaled one times it, up to rounding."""
    geom, w, hip, _ = decoders[name]
    s = np.float32(2.0) ** exponent
    ws = {k: v * s if k.startswith(("dec.conv_pre.", "dec.cond.", "dec.noise_convs."))
          or (k.startswith(("dec.ups.", "dec.resblocks.")) and k.endswith(".bias")) else v for k, v in w.items()}
    scaled = HipSynthesizer(ws, sr=geom.sr)
    P = 70
    d = syn.make_dec_inputs(geom, P, seed=3)
    for m in (hip, scaled):
        m.set_debug(True)
        m.dec.forward(d["z"], d["f0"], d["g"], d["ns"])
        m.set_debug(False)
    for i, c in enumerate(geom.stage_channels()):
        shape = (1, c, P * 2 ** (i + 1))
        assert rel_l2(scaled.read(f"dec_stage{i}", shape) / s, hip.read(f"dec_stage{i}", shape)) < 2e-6
    scaled.close()


@pytest.mark.parametrize("name", sorted(GEOMS))
def test_infinity_reaches_what_it_reaches_in_fp32(decoders, name):
    """An infinite value of z: the samples it does not reach are unchanged, and
    what is NaN in the fp32 path is NaN."""
    geom, _, hip, ref = decoders[name]
    P = 300
    d = syn.make_dec_inputs(geom, P, seed=9)
    z = d["z"].copy()
    z[0, 5, 150] = np.inf
    with nn_ref.conv_formulation("taps"), np.errstate(all="ignore"):
        want = ref.forward(z, d["f0"], d["g"], d["ns"])
        clean = ref.forward(d["z"], d["f0"], d["g"], d["ns"])
    got = hip.dec.forward(z, d["f0"], d["g"], d["ns"])
    fine = np.isfinite(want) & (np.abs(want - clean) < 1e-6)
    assert fine.any() and not fine.all()
    assert np.abs(got[fine] - want[fine]).max() < 1e-4
    assert np.isnan(got[np.isnan(want)]).all()


@pytest.mark.parametrize("name,P,exponent", [(n, P, e) for n in sorted(GEOMS) for P, e in
                                             ((700, 24), (700, 60), (700, 100), (3000, 60), (9000, 60))])
def test_a_spike_takes_nothing_from_its_neighbours(decoders, name, P, exponent):
    """The samples that frames of huge or infinite z do not reach share tiles with
    those they do, and keep their fp32 precision: what is computed twice, with
    and without the spikes, differs by the error of two such computations."""
    geom, _, hip, ref = decoders[name]
    d = syn.make_dec_inputs(geom, P, seed=9)
    z, zi = d["z"].copy(), d["z"].copy()
    z[0, :, 70::160] = np.float32(2.0) ** exponent
    zi[0, :, 70::160] = np.inf
    with nn_ref.conv_formulation("taps"), np.errstate(all="ignore"):
        reach = ref.forward(zi, d["f0"], d["g"], d["ns"])
        clean = ref.forward(d["z"], d["f0"], d["g"], d["ns"])
    fine = np.abs(reach - clean) < 1e-6
    assert 0.1 < fine.mean() < 0.9
    want = hip.dec.forward(d["z"], d["f0"], d["g"], d["ns"])
    for x in (z, zi):
        got = hip.dec.forward(x, d["f0"], d["g"], d["ns"])
        assert rel_l2(got[fine], want[fine]) < 3e-6


@pytest.mark.parametrize("name,P", [("fused", P) for P in (1, 17, 64, 129, 2100, 8400, 16900)] +
                         [("plain", P) for P in (1, 33, 1601, 4300)])
def test_bf16_tile_edges(decoders, name, P):
    """ResBlocks on bf16 operands: rounding two operands of every product gives
    2^-9 sqrt(2 / 3) per conv, about 7e-3 over 18 of them; no sample is off by
    more than a dozen times that."""
    geom, w, hip, _ = decoders[name]
    bf = HipSynthesizer(w, sr=geom.sr, precision=2)
    d = syn.make_dec_inputs(geom, P, seed=P)
    want = hip.dec.forward(d["z"], d["f0"], d["g"], d["ns"])
    got = bf.dec.forward(d["z"], d["f0"], d["g"], d["ns"])
    bf.close()
    assert 1e-4 < rel_l2(got, want) < 1.4e-2
    assert np.abs(got - want).max() < 0.084 * np.sqrt((want ** 2).mean())
