"""The f16 pair hi + lo that a normed activation is multiplied as is the pair of its f32 value.

The product of a residual value and its norm weight goes to f16 twice: as the stored hi, and in the difference
that lo is. Rounded once from the exact product in one place and from the rounded f32 product in the other,
hi differs where the f32 product is halfway between two f16 values, and the pair is off by a whole f16 unit. Here
every residual value is such a one: with hi taken two ways, V (the first layer's values, a plain
projection) is off by about 1e-3 and hardly one f16 value in three is right. Otherwise two correct f32 sums of
1024 products differ by about 1e-6 of the value, 1e-6 / 2^-11 = 0.2 % of the f16 roundings: 2 % allowed.
"""
import numpy as np
import pytest

from gpu_util import log

pytestmark = pytest.mark.gpu

W = np.float32(1.1)


def _halfway_rows(T):
    """Values whose exact product with W is rounded to a tie of f16 in f32, from the side that the
    even neighbour does not lie on."""
    t = 1 + (2 * np.arange(1024) + 1) * 2.0 ** -11           # the midpoints of f16 in [1, 2)
    x = (t / np.float64(W)).astype(np.float32)
    exact = x.astype(np.float64) * np.float64(W)             # 48 bits: exact
    f32 = exact.astype(np.float32)
    twice, once = f32.astype(np.float16).astype(np.float64), np.where(exact > t, t + 2.0 ** -11, t - 2.0 ** -11)
    x = x[(f32 == t) & (exact != t) & (twice != once)]
    assert len(x) > 100
    rng = np.random.default_rng(T)
    return (rng.choice(x, (T, 1024)) * rng.choice([-1.0, 1.0], (T, 1024))).astype(np.float32)


@pytest.fixture(scope="module")
def side(scratch_dir):
    from navi_amd import abi, blob
    from oracle.model import Oracle
    path = scratch_dir / "pairs.navi"
    kv = blob.qwen3tts_0p6b_kv(talker_layers=1, cp_layers=1, text_vocab=64)
    blob.write_navi(path, kv, blob.tensor_table(kv, ("talker", "cp")), 6,
                    {"talker.model.layers.0.input_layernorm.weight": np.full(1024, W, np.float32)})
    abi.device_open()
    weights = abi.DeviceWeights(path, select=lambda t: t.name.startswith("talker."))
    t = abi.Talker(weights, 512, 600)
    yield abi, t, Oracle(path)
    t.close()
    path.unlink()


# the row kernels' tiles (10, 32, 48, 64 rows) and the streamed projections' (65, 130, 300, 500)
@pytest.mark.parametrize("T", [10, 32, 48, 64, 65, 130, 300, 500])
def test_values_of_halfway_products(side, T):
    abi, t, ora = side
    rows = _halfway_rows(T)
    d = abi.DeviceBuffer(rows.nbytes)
    d.upload(rows)
    t.prefill(d.ptr, T)
    kvo = ora.new_kv(T + 1)
    ora.prefill(rows, kvo)
    got, want = t.kv.read(0, T)[1], kvo[0][1][:T].numpy()
    off = float(np.mean(got != want))
    log(f"  T={T}: {off:.4f} of the values differ")
    assert off < 0.02
