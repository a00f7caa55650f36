"""A row's results do not depend on how many rows a prompt has: every projection adds the same products in
the same order at every row count, so the rows of a longer prompt are a shorter one's bit for bit.

Up to 64 rows the whole-K row kernels share their tiles between blocks by the row count (rows.h): the
reference is the 10-row prompt. From there to 256 rows it is the 64-row prompt, the most those kernels
take: above it the streamed projections (gemm.h) and the attention that reads the cache have to give its
bits. Above 256 rows the attention is the matrix cores' in 256-key chunks, with bits of its own from the
second layer on: the reference is the 257-row prompt there, and the 64-row one for the first layer's
keys and values.
"""
import numpy as np
import pytest

from gpu_util import compare, log

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def side(small_blob):
    from navi_amd import abi
    from oracle.model import Oracle
    abi.device_open()
    W = abi.DeviceWeights(small_blob, select=lambda t: t.name.startswith("talker."))
    t = abi.Talker(W, 2048, 2100)
    rows = np.random.default_rng(1).standard_normal((2056, 1024)).astype(np.float32)
    d = abi.DeviceBuffer(rows.nbytes)
    d.upload(rows)
    ora = Oracle(small_blob)

    def prefill(T):
        t.prefill(d.ptr, T)
        return [t.kv.read(l, T) for l in range(ora.tp.n_layer)]
    yield prefill, t, ora, rows, {n: prefill(n) for n in (10, 64, 257)}
    t.close()


def _same(got, want, layers, n):
    for l in layers:
        for a, b in zip(got[l], want[l]):
            np.testing.assert_array_equal(a[:n], b[:n])


@pytest.mark.parametrize("T", [16, 17, 32, 33, 48, 49, 64])
def test_shared_tiles_have_the_same_bits(side, T):
    prefill, _, ora, _, want = side
    _same(prefill(T), want[10], range(ora.tp.n_layer), 10)


# every tile choice of the streamed projections (gemm.h's launch rules), its first and last row counts
@pytest.mark.parametrize("T", [65, 80, 81, 128, 129, 160, 161, 200, 240, 256])
def test_rows_have_the_row_kernels_bits(side, T):
    prefill, _, ora, _, want = side
    _same(prefill(T), want[64], range(ora.tp.n_layer), 64)


@pytest.mark.parametrize("T", [300, 320, 321, 384, 385, 512, 513, 640, 641, 768, 769, 1001, 1025, 2056])
def test_long_prompts_rows_are_the_shorter_ones(side, T):
    prefill, _, ora, _, want = side
    got = prefill(T)
    _same(got, want[64], [0], 64)
    _same(got, want[257], range(ora.tp.n_layer), 257)


def test_longest_prompt_matches_oracle(side):
    """A prompt past 1032 rows, the reference's maximum, up to which the other files go."""
    prefill, t, ora, rows, _ = side
    T = 2050
    got = prefill(T)
    hid, lg = t.hidden_logits()
    kvo = ora.new_kv(T + 1)
    ohid, olg = ora.prefill(rows[:T], kvo)
    for name, g, w in (("hidden", hid, ohid), ("logits", lg, olg)):
        mx, cos = compare(g, w)
        log(f"  T={T} {name}: max abs {mx:.3e} cosine {cos:.7f}")
        assert mx < 2e-2 and cos > 0.9995
    for l, kv in enumerate(got):
        for g, w in zip(kv, kvo[l]):
            assert np.allclose(g, w[:T].numpy(), rtol=4e-3, atol=2e-3)
