"""The speaker encoder's time reductions (SE mean, pooling statistics with their softmax over time) and
its Res2Net chains at the edges of their row splits, against the CPU oracle.

A thread takes rows q, q + 64, ... and keeps 16 of them: fewer rows than slices, one row more than whole
slices, the last length in registers (1024), the first read again (1025), a third pass (2100). A
chain's block owns 16 rows and computes up to 24 more on either side (dilations 2, 3, 4), mirrored at
the ends: less than a block, whole blocks and a ragged row, halos that reach both ends of the audio
(5 .. 33), one end (40, 41) and neither.
Tolerance: both sides hold f32 and sum at most 4608 terms at a time, sqrt(4608) 2^-24 = 4e-6 of
the sum's scale for rounding errors of random sign; five times that for the chain of layers.
"""
import numpy as np
import pytest

from gpu_util import log

pytestmark = pytest.mark.gpu

REL = 2e-5


@pytest.fixture(scope="module")
def spk(speaker_blob):
    from navi_amd import abi
    from oracle.speaker import SpeakerOracle
    abi.device_open()
    W = abi.DeviceWeights(speaker_blob, select=lambda t: t.name.startswith("speaker_encoder."))
    return abi.Speaker(W, max_seconds=30.0), W, SpeakerOracle(speaker_blob)


@pytest.mark.parametrize("T", [5, 63, 64, 65, 128, 129, 1024, 1025, 2100])
def test_reductions_match_oracle(spk, T):
    check(spk, T)


@pytest.mark.parametrize("T", [6, 15, 16, 17, 31, 32, 33, 40, 41, 95])
def test_res2net_chains_match_oracle(spk, T):
    check(spk, T)


def check(spk, T):
    s, _, ora = spk
    mel = np.random.default_rng(T).normal(-4.0, 2.0, (128, T)).astype(np.float32)
    got, want = np.asarray(s.embed_mel(mel), np.float64), np.asarray(ora.embed_mel(mel), np.float64)
    rel = float(np.sqrt(np.mean((got - want) ** 2) / np.mean(want ** 2)))
    log(f"  {T} frames: rel rms {rel:.2e}")
    assert np.isfinite(got).all() and rel <= REL
    assert np.array_equal(s.embed_mel(mel), s.embed_mel(mel))
