"""Prefills above the row kernels' 64 rows (gemm.h) at the edges of their tile choice, their f16-range
flag and their query scale, against the CPU oracle (Talker::prefill, talker.hip:354-399).

Tolerances: the hidden and logits bars of the other prefill tests; K/V rows are f16, so two correct
results differ by at most a rounding step or two (2^-9 relative, here 4e-3) where an f32 sum in another
order falls on the other side of one.
"""
import numpy as np
import pytest

from gpu_util import compare, log

pytestmark = pytest.mark.gpu

TOL_ABS, TOL_COS = 2e-2, 0.9995


class Side:
    def __init__(self, path):
        from navi_amd import abi
        from oracle.model import Oracle
        abi.device_open()
        self.abi, self.ora = abi, Oracle(path)
        self.W = abi.DeviceWeights(path, select=lambda t: t.name.startswith("talker."))
        self.talker = abi.Talker(self.W, 1024, 1100)

    def prefill(self, rows):
        d = self.abi.DeviceBuffer(rows.nbytes)
        d.upload(rows)
        self.talker.prefill(d.ptr, rows.shape[0])
        hid, lg = self.talker.hidden_logits()
        kv = [self.talker.kv.read(l, rows.shape[0]) for l in range(self.ora.tp.n_layer)]
        d.free()
        return hid.copy(), lg.copy(), kv

    def check(self, rows):
        hid, lg, kv = self.prefill(rows)
        T = rows.shape[0]
        kvo = self.ora.new_kv(T + 1)
        ohid, olg = self.ora.prefill(rows, kvo)
        for name, got, want in (("hidden", hid, ohid), ("logits", lg, olg)):
            mx, cos = compare(got, want)
            log(f"  T={T} {name}: max abs {mx:.3e} cosine {cos:.7f}")
            assert mx < TOL_ABS and cos > TOL_COS
        for l, (k, v) in enumerate(kv):
            for got, want in ((k, kvo[l][0][:T].numpy()), (v, kvo[l][1][:T].numpy())):
                assert np.allclose(got, want, rtol=4e-3, atol=2e-3)
                assert np.mean(got != want) < 0.05


@pytest.fixture(scope="module")
def side(small_blob):
    s = Side(small_blob)
    yield s
    s.talker.close()


def _rows(T):
    return np.random.default_rng(T).standard_normal((T, 1024)).astype(np.float32)


# the last row count of one tile choice and the first of the next: gate|up 80, 128, 160, 256, 512; q|k|v
# 128, 256, 384, 512, 768; o and down 128, 256, 512 (65, 256, 257, 512 and 513 are in
# test_prefill_gpu.py); 96: an even number of 16-row tiles with no ragged row
@pytest.mark.parametrize("T", [66, 80, 81, 96, 128, 129, 160, 161, 384, 385, 768, 769])
def test_prefill_tile_edges_match_oracle(side, T):
    side.check(_rows(T))


@pytest.mark.parametrize("T", [65, 300])
def test_prefill_out_of_range_activation(side, T):
    """A residual row times the norm weight outside f16 is an error, and the next call starts clean."""
    rows = _rows(T)
    want = side.prefill(rows)
    bad = rows.copy()
    bad[T - 2, 5] = 1e5
    with pytest.raises(side.abi.NaviError, match="f16 range"):
        side.prefill(bad)
    got = side.prefill(rows)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
    for (gk, gv), (wk, wv) in zip(got[2], want[2]):
        np.testing.assert_array_equal(gk, wk)
        np.testing.assert_array_equal(gv, wv)


def test_prefill_large_query_norm(scratch_dir):
    """Query norm weights whose queries leave the f16 range: held scaled by a power of two."""
    from navi_amd import blob
    path = scratch_dir / "large_q.navi"
    kv = blob.qwen3tts_0p6b_kv(talker_layers=1, cp_layers=1, text_vocab=64)
    w = np.full(128, 7000.0, np.float32)
    blob.write_navi(path, kv, blob.tensor_table(kv, ("talker", "cp")), 5,
                    {"talker.model.layers.0.self_attn.q_norm.weight": w})
    s = Side(path)
    try:
        s.check(_rows(70))
    finally:
        s.talker.close()
        path.unlink()
