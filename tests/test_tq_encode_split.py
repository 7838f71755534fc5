"""TurboQuant encode on the matrix cores (eos_tq_encode_split_*): codes and
norms bit-exact against the CPU oracle at the edges of its tiles (96 vectors,
32 coordinates per wavefront, 4 / 8 / 12 wavefronts, several blocks of
coordinates), with and without 16-byte rows, and for vectors its error bound
leaves to the exact decision: ties, zero vectors, norms out of the range of
the split, infinities and NaN."""
import numpy as np
import pytest

import oracle
from eos_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from eos_amd.runtime import Runtime
    r = Runtime(0)
    yield r
    r.close()


def _check(rt, x, rot, d, bits):
    from eos_amd.turboquant import TurboQuantIndex
    cb, s = datagen.turboquant_codebook(bits, d)
    rb = (d * bits + 7) // 8
    tq = TurboQuantIndex(rt, np.zeros((0, rb), np.uint8), np.zeros(0, np.float32), d, bits, cb, s,
                         rot)
    codes, norms = tq.encode(x)
    want_c, want_n = oracle.tq_encode(x, rot, d, bits, cb, s)
    np.testing.assert_array_equal(norms, want_n)
    np.testing.assert_array_equal(codes, want_c)
    tq.release()


@pytest.mark.parametrize("d,bits,n", [(1, 4, 3), (31, 2, 95), (32, 4, 96), (33, 4, 97),
                                      (128, 2, 191), (129, 4, 193), (256, 4, 200), (383, 4, 97),
                                      (384, 2, 769), (385, 4, 100), (513, 2, 97), (768, 4, 96),
                                      (1023, 4, 65), (1024, 2, 98)])
def test_encode_split_bit_exact(rt, d, bits, n):
    print(f"[case] split encode d={d} bits={bits} n={n}", flush=True)
    x = datagen.normal(d + n, n * d).astype(np.float32).reshape(n, d)
    x *= np.exp(datagen.normal(d, n) * 3)[:, None].astype(np.float32)
    _check(rt, x, datagen.orthogonal(d + 7, d).astype(np.float32), d, bits)


@pytest.mark.parametrize("d", [96, 130, 384])
def test_encode_split_undecided_vectors(rt, d):
    """A signed permutation as rotation makes every coordinate of a one-hot
    or constant vector a tie or equal; norms of 0, 2^-110, 2^110, infinity
    and NaN; 98 such rows fill one tile's list over and leave a second tile."""
    print(f"[case] split encode undecided d={d}", flush=True)
    perm = np.argsort(datagen.uniform(d, d))
    rot = np.zeros((d, d), np.float32)
    rot[np.arange(d), perm] = np.where(np.arange(d) % 2 == 0, 1.0, -1.0)
    x = np.zeros((98, d), np.float32)
    x[np.arange(60), np.arange(60) % d] = 1.5
    x[60:90] = datagen.normal(d + 1, 30 * d).astype(np.float32).reshape(30, d)
    x[62] *= np.float32(2.0 ** -110)
    x[63] *= np.float32(2.0 ** 110)
    x[64, 3] = np.inf
    x[65, 4] = np.nan
    x[66, :] = 0.25
    with np.errstate(all="ignore"):
        _check(rt, x, rot, d, 4)
        _check(rt, x[58:70], datagen.orthogonal(d + 9, d).astype(np.float32), d, 2)


@pytest.mark.parametrize("d,bits", [(1, 4), (16, 4), (33, 2), (47, 4), (100, 2), (130, 4), (384, 4),
                                    (385, 4), (770, 2), (1024, 4)])
def test_encode_split_ties(rt, d, bits):
    """Zeros under a signed permutation are exact ties of the symmetric
    levels: few of them (a thread's chains each), too many for a tile's list
    (the whole tile on f64 MFMA), and a tile of tiny vectors, which leave
    every coordinate to the list."""
    print(f"[case] split encode ties d={d} bits={bits}", flush=True)
    rng = np.random.default_rng(d)
    rot = np.zeros((d, d), np.float32)
    rot[np.arange(d), rng.permutation(d)] = np.where(np.arange(d) % 2 == 0, 1.0, -1.0)
    x = rng.normal(size=(3 * 96 + 50, d)).astype(np.float32)
    x[:96][rng.random((96, d)) < 0.01] = 0
    x[96:192][rng.random((96, d)) < 0.6] = 0
    x[192:288] *= np.float32(1e-31)
    x[288:, : (d + 1) // 2] = 0
    with np.errstate(all="ignore"):
        x[200, 0], x[201, d - 1], x[202] = np.inf, np.nan, 0
        _check(rt, x, rot, d, bits)
        _check(rt, x[192:230], datagen.orthogonal(d + 9, d).astype(np.float32), d, bits)
