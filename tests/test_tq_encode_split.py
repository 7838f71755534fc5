"""TurboQuant encode on the matrix cores (eos_tq_encode_split_*): codes and
norms bit-exact against the CPU oracle at the edges of its tiles (96 vectors,
32 coordinates per wavefront, 4 / 8 / 12 wavefronts, several blocks of
coordinates), with and without 16-byte rows, and for vectors its error bound
leaves to the exact decision: ties, zero vectors, norms out of the range of
the split, infinities and NaN; next to decision points for sums whose every
rounding goes the same way; with levels out of order and repeated; and by the
f64 kernels, which scales outside the split's bound and quantizers without a
rotation take."""
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


def _check(rt, x, rot, d, bits, levels=None):
    from eos_amd.turboquant import TurboQuantIndex
    cb, s = levels or datagen.turboquant_codebook(bits, d)
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


def _lossy(v, rng):
    """Positive values near v whose bf16 pair leaves out as much as it can."""
    def bf16(a):
        u = a.astype(np.float32).view(np.uint32).astype(np.uint64)
        return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)
    high = bf16(v)
    low = bf16(high * np.float32(2.0 ** -9) * rng.uniform(0.55, 0.95, v.shape).astype(np.float32))
    return ((high.astype(np.float64) + low) * (1 + 2.0 ** -17.3)).astype(np.float32)


@pytest.mark.parametrize("d,spiked", [(32, False), (64, True), (384, False), (384, True),
                                      (768, True)])
def test_encode_split_next_to_decision_points(rt, d, spiked):
    """Rows and vectors of positive terms (so that u is about |R_j| |x| and
    every part the split drops or rounds away lowers it), each vector moved by
    a free coordinate until one u_j lies within two error bounds of a decision
    point: pairs just inside the bound are decided in f64, those just outside
    by the split product."""
    print(f"[case] split encode at decision points d={d} spiked={spiked}", flush=True)
    rng = np.random.default_rng(d)
    n, bits = 96 * 4, 4
    levels = np.linspace(-127, 127, 16).round().astype(np.int8)
    scale = float(np.float32(1 / 127))
    points = np.array(sorted({int(a) + int(b) for a, b in zip(levels, levels[1:])})) * scale / 2

    def terms(*shape):
        if not spiked:
            return rng.uniform(1.0, 1.9, shape)
        m = np.exp2(rng.uniform(-9, -7, shape))
        m[..., ::32] = 1.0
        return m

    rot = (rng.normal(size=(d, d)) * 0.02 / np.sqrt(d)).astype(np.float32)
    rows = rng.choice(d, 6, replace=False)
    for j in rows:
        r = terms(d)
        rot[j] = _lossy((r / np.linalg.norm(r)).astype(np.float32), rng)
    x = _lossy(terms(n, d).astype(np.float32), rng)
    free = d // 3
    rot[:, free] = 0
    x[:, free] = 0
    pick = rows[rng.integers(0, len(rows), n)]
    x64, r64 = x.astype(np.float64), rot[pick].astype(np.float64)
    u, ss = (x64 * r64).sum(1), (x64 * x64).sum(1)
    point = np.array([points[points < c - 1e-4].max() for c in u / np.sqrt(ss)])
    bound = 1.7e-5  # of |u~ - u| / |x|, the largest of these dimensions
    target = point + rng.uniform(-2, 2, n) * bound
    x[:, free] = np.sqrt((u / target) ** 2 - ss).astype(np.float32)
    x64 = x.astype(np.float64)
    near = np.abs((x64 * r64).sum(1) / np.linalg.norm(x64, axis=1) - point) < 2.1 * bound
    assert near.all()
    _check(rt, x, rot, d, bits, (levels, scale))


@pytest.mark.parametrize("d,bits", [(96, 4), (384, 4), (130, 2)])
def test_encode_split_unsorted_and_repeated_levels(rt, d, bits):
    """Levels out of order, and two codes of one level: the lower code wins."""
    print(f"[case] split encode levels d={d} bits={bits}", flush=True)
    rng = np.random.default_rng(bits)
    levels = np.linspace(-100, 90, 1 << bits).round().astype(np.int8)
    rng.shuffle(levels)
    levels[-1] = levels[0]
    levels[1] = levels[2]
    x = rng.normal(size=(200, d)).astype(np.float32)
    x[7] = 0
    rot = datagen.orthogonal(d + 3, d).astype(np.float32)
    scale = float(np.float32(2.5 / np.sqrt(d) / 100))
    _check(rt, x, rot, d, bits, (levels, scale))
    _check(rt, x, rot, d, bits, (np.full(1 << bits, 5, np.int8), scale))


@pytest.mark.parametrize("d,bits,why", [(384, 4, "scale"), (700, 2, "scale"), (384, 4, "large"),
                                        (700, 4, "large"), (96, 2, "small"), (384, 4, "unrotated"),
                                        (513, 2, "unrotated"), (1024, 4, "unrotated")])
def test_encode_outside_the_split(rt, d, bits, why):
    """The f64 kernels (dims up to 512 and up to 1,024): a level scale below
    the split's resolution, rotation rows above 2^20 and below 2^-20, and no
    rotation."""
    print(f"[case] f64 encode d={d} bits={bits} {why}", flush=True)
    x = datagen.normal(d + bits, 77 * d).astype(np.float32).reshape(77, d)
    x[5] = 0
    rot = None
    cb, s = datagen.turboquant_codebook(bits, d)
    if why != "unrotated":
        rot = datagen.orthogonal(d + 5, d).astype(np.float32)
        factor = {"scale": 1.0, "large": 2.0 ** 21, "small": 2.0 ** -22}[why]
        rot = rot * np.float32(factor)
        s = float(np.float32(s * (1e-4 if why == "scale" else factor)))
    _check(rt, x, rot, d, bits, (cb, s))
