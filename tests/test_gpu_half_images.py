"""Prompts and chunks over IEEE-half and E4M3 caches run on tile images without lo halves.
They must give the bits of the three-product path over an f32 cache that holds the same
values: the products left out are products with zeros."""
import numpy as np
import pytest

import eyebrowse_amd as eb
import oracle
from tests._gpu import assert_bitwise, note, upload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return eb.Device.new(0)


def _chunk(dev, q, kc, vc, dtype, h, hkv, pos0, rows, hd, max_seq, scale, window):
    qt = upload(dev, q)
    ot = eb.Tensor.empty(dev, (rows, h, hd))
    kt, vt = (eb.Tensor.empty(dev, (max_seq, hkv, hd), dtype) for _ in range(2))
    rec = eb.Recorder(dev)
    for t, x in ((kt, kc), (vt, vc)):
        eb.kv_write(rec, t, upload(dev, x), hkv, max_seq, hd, max_seq, 0)
    eb.attn_prefill_chunk(rec, qt, kt, vt, ot, h, hkv, pos0, rows, hd, max_seq, scale, window)
    rec.submit()
    return ot.to_f32()


@pytest.mark.parametrize("dtype", [eb.DType.F16, eb.DType.F8E4M3])
@pytest.mark.parametrize("h,hkv,hd,pos0,rows,window", [
    (4, 2, 32, 31, 5, 0),       # one block: staged, smallest split head dim
    (4, 2, 64, 1, 130, 0),      # three blocks: records
    (8, 2, 128, 33, 33, 0),     # GQA 4, two blocks: staged, a tile's remainder
    (8, 2, 128, 65, 129, 40),   # GQA 4, records, windowed
    (2, 2, 80, 7, 300, 0),      # GQA 1, padded head dim, records
    (4, 2, 256, 3, 64, 0),      # one block at 256: staged
    (4, 2, 256, 95, 97, 0),     # two blocks at 256: records
    (128, 8, 128, 10, 545, 0),  # more than 512 blocks of 4 heads: records without a key split
    (128, 8, 128, 70, 530, 90),  # the same, windowed
    (64, 16, 64, 0, 1030, 0),   # the same at 64, from position 0
])
def test_same_bits_as_f32_cache(dev, dtype, h, hkv, hd, pos0, rows, window):
    note(f"half images {dtype.name} hd={hd} pos0={pos0} rows={rows} window={window}")
    keys = pos0 + rows
    q = oracle.randn((rows, h, hd), 1)
    kc, vc = oracle.randn((keys, hkv, hd), 2), oracle.randn((keys, hkv, hd), 3)
    vc[keys // 2] *= 100.0   # (E4M3's largest value is 448)
    kc[0] *= 2.0 ** -9       # E4M3 subnormals
    vc[1] *= 2.0 ** -20      # half subnormals, E4M3 zeros
    if dtype == eb.DType.F16:
        kr, vr = (x.astype(np.float16).astype(np.float32) for x in (kc, vc))
    else:
        kr, vr = (oracle.f8_values(oracle.f8_bits(x)).reshape(x.shape) for x in (kc, vc))
    args = (h, hkv, pos0, rows, hd, keys, 0.1, window)
    got = _chunk(dev, q, kc, vc, dtype, *args)
    want = _chunk(dev, q, kr, vr, eb.DType.F32, *args)
    assert_bitwise(got, want, "half images against split images")


def test_infinities_as_f32_cache(dev):
    """Infinities and NaN of a half cache reach the same outputs as through the split path."""
    note("half images with infinities")
    h, hkv, hd, pos0, rows = 8, 2, 128, 10, 200
    keys = pos0 + rows
    q = oracle.randn((rows, h, hd), 4)
    kc, vc = oracle.randn((keys, hkv, hd), 5), oracle.randn((keys, hkv, hd), 6)
    kc, vc = (x.astype(np.float16).astype(np.float32) for x in (kc, vc))
    vc[100, 0, 3], vc[120, 1, 7], kc[150, 0, 9] = np.inf, np.nan, -np.inf
    args = (h, hkv, pos0, rows, hd, keys, hd ** -0.5, 0)
    got = _chunk(dev, q, kc, vc, eb.DType.F16, *args)
    want = _chunk(dev, q, kc, vc, eb.DType.F32, *args)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])
