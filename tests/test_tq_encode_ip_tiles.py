"""The inner-product encode on the f64 matrix cores: codes, signs, ResNorm and
Norm bit-exact against the CPU oracle at the edges of its tiles (16 rows and
vectors, 128 coordinates per kernel variant, 64-wide K chunks), with zero,
infinite and NaN vectors and exact ties. Calls of up to 16 vectors a CU and
dims up to 512 run eos_tq_encode_ip_s* (16 vectors per workgroup), others
eos_tq_encode_ip_t* (32, above dim 512 16)."""
import numpy as np
import pytest

import oracle
from eos_amd.turboquant import IPQuantizer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,bits,n,rotate", [(1, 1, 2, True), (16, 4, 31, True), (17, 3, 33, True),
                                             (64, 2, 32, True), (65, 1, 64, True),
                                             (127, 3, 40, False), (128, 4, 33, True),
                                             (129, 3, 65, True), (255, 2, 32, True),
                                             (257, 4, 35, True), (385, 3, 33, True),
                                             (512, 4, 40, True), (513, 3, 17, True),
                                             (640, 1, 16, True), (700, 2, 20, False),
                                             (897, 3, 18, True), (1024, 4, 17, True)])
def test_encode_ip_tiles_bit_exact(rt, d, bits, n, rotate):
    print(f"[case] ip encode d={d} bits={bits} n={n} rotate={rotate}", flush=True)
    rng = np.random.default_rng(d * 31 + bits)
    rot = np.linalg.qr(rng.normal(size=(d, d)))[0].astype(np.float32) if rotate else None
    S = rng.normal(size=(d, d)).astype(np.float32)
    cb = np.linspace(-127, 127, 1 << bits).round().astype(np.int8)
    s_c = float(np.float32(2.5 / np.sqrt(d) / 127))
    x = rng.normal(size=(n, d)).astype(np.float32)
    x[0] = 0
    x[1] = 0
    x[1, d // 2] = 2.0  # zeros among the coordinates: ties without a rotation
    x[n - 1] *= np.float32(1e-30)
    if n > 16:
        x[5, 0] = np.inf
        x[6, d - 1] = np.nan
        x[16] *= np.float32(1e30)
    iq = IPQuantizer(rt, d, bits, cb, s_c, rot, S)
    with np.errstate(all="ignore"):
        got = iq.encode(x)
        want = oracle.tq_encode_ip(x, rot, S, d, bits, cb, s_c)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
    iq.release()


@pytest.mark.parametrize("d,bits", [(24, 2), (130, 3), (300, 1), (512, 4), (520, 3), (1000, 2)])
def test_encode_ip_large_calls_equal_small_ones(rt, d, bits):
    """Calls above 16 vectors a CU take workgroups of 32 vectors (16 above dim
    512) and shorter loads; the same vectors in calls of 1,111 do not."""
    n = 16 * 256 + 37
    print(f"[case] ip encode large d={d} bits={bits} n={n}", flush=True)
    rng = np.random.default_rng(d + bits)
    rot = np.linalg.qr(rng.normal(size=(d, d)))[0].astype(np.float32)
    S = rng.normal(size=(d, d)).astype(np.float32)
    cb = np.linspace(-127, 127, 1 << bits).round().astype(np.int8)
    x = rng.normal(size=(n, d)).astype(np.float32)
    x[4100] = 0
    qz = IPQuantizer(rt, d, bits, cb, float(np.float32(2.5 / np.sqrt(d) / 127)), rot, S)
    whole = qz.encode(x)
    parts = [qz.encode(x[i:i + 1111]) for i in range(0, n, 1111)]
    for w, *p in zip(whole, *parts):
        np.testing.assert_array_equal(w, np.concatenate(p))


@pytest.mark.parametrize("d,bits,rotate", [(96, 3, False), (200, 3, True), (384, 3, True),
                                           (512, 2, False), (640, 4, True), (768, 3, True),
                                           (800, 2, True), (1024, 1, False)])
def test_encode_ip_large_calls_match_oracle(rt, d, bits, rotate):
    """eos_tq_encode_ip_t* of every width: zero, infinite, NaN and one-hot
    vectors in the first and in the last, partial workgroup against the
    oracle, all others against the same vectors in small calls."""
    n = 16 * rt.info()["compute_units"] + 41
    print(f"[case] ip encode large against oracle d={d} bits={bits} n={n}", flush=True)
    rng = np.random.default_rng(d + 7 * bits)
    rot = np.linalg.qr(rng.normal(size=(d, d)))[0].astype(np.float32) if rotate else None
    S = rng.normal(size=(d, d)).astype(np.float32)
    cb = np.linspace(-127, 127, 1 << bits).round().astype(np.int8)
    s_c = float(np.float32(2.5 / np.sqrt(d) / 127))
    x = rng.normal(size=(n, d)).astype(np.float32)
    for i in (0, n - 9):
        x[i:i + 2] = 0
        x[i + 1, d // 2] = 2.0
        x[i + 2, 0] = np.inf
        x[i + 3, d - 1] = np.nan
        x[i + 4] *= np.float32(1e-30)
        x[i + 5] *= np.float32(1e30)
    iq = IPQuantizer(rt, d, bits, cb, s_c, rot, S)
    edge = np.r_[0:34, n - 43:n]
    with np.errstate(all="ignore"):
        whole = iq.encode(x)
        want = oracle.tq_encode_ip(x[edge], rot, S, d, bits, cb, s_c)
        parts = [iq.encode(x[i:i + 1000]) for i in range(0, n, 1000)]
    for w, o, *p in zip(whole, want, *parts):
        np.testing.assert_array_equal(w[edge], o)
        np.testing.assert_array_equal(w, np.concatenate(p))
    iq.release()
