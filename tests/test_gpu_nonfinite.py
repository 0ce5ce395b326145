# -*- coding: utf-8 -*-
"""Calls whose every sum is NaN: the split kernels form such sums again on the
fp32 matrix cores.  They return NaN, and in a time of the order of a finite
call's (about 16 / 3 of the split products' for the convolutions alone, at the
rates of the two instructions, and the finite call's own on top; 12 leaves room
for tiles too few to fill the card)."""

from __future__ import annotations

import time

import numpy as np
import pytest

from rvc_hip import synthetic as syn
from rvc_hip.hubert import HipHubert
from rvc_hip.pipeline import HipVcGlue
from rvc_hip.synth import HipSynthesizer

pytestmark = pytest.mark.gpu


def _best(call):
    best = np.inf
    for _ in range(4):
        t0 = time.perf_counter()
        out = call()
        best = min(best, time.perf_counter() - t0)
    return best, out


def _compare(call, x):
    finite, _ = _best(lambda: call(x))
    nan, out = _best(lambda: call(np.full_like(x, np.nan)))
    print(f"finite {finite * 1e3:.2f} ms, NaN {nan * 1e3:.2f} ms", flush=True)
    assert nan < 12 * finite
    return out


# stage channels 128 / 64 / 32 (a dilation group a launch) and 192 / 96 (a launch per conv)
@pytest.mark.parametrize("initial,n_ups", [(256, 3), (384, 2)])
def test_decoder(initial, n_ups):
    geom = syn.Geometry(phone_dim=64, hidden=48, filter_channels=96, n_layers=1, gin=32, n_spk=2,
                        upsample_initial=initial, upsample_rates=(2,) * n_ups, upsample_kernels=(4,) * n_ups,
                        sr=100 * 2 ** n_ups)
    m = HipSynthesizer(syn.make_weights(geom, seed=4), sr=geom.sr)
    d = syn.make_dec_inputs(geom, 3000, seed=1)
    y = _compare(lambda z: m.dec.forward(z, d["f0"], d["g"], d["ns"]), d["z"])
    m.close()
    assert np.isnan(y).all()


def test_hubert():
    m = HipHubert(syn.make_hubert_weights(syn.HUBERT_BASE, seed=6))
    y = _compare(m.encode, syn.make_hubert_input(64000, seed=1))
    m.close()
    assert np.isnan(y).all()


def test_search():
    r = np.random.default_rng(2)
    glue = HipVcGlue()
    glue.set_index(r.standard_normal((5000, 768), dtype=np.float32))
    _compare(lambda q: glue.search(q)[0], r.standard_normal((200, 768), dtype=np.float32))
