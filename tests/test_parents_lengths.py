"""Parents by a lane (up to 64 children) and by a wavefront (more), alone and
mixed, and the chunked ranking of parent scores: ids, scores and best children
bit-exact against the CPU oracle."""
import numpy as np
import pytest

import oracle
from eos_amd import datagen

pytestmark = pytest.mark.gpu


def _offsets(counts):
    return np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)


@pytest.mark.parametrize("name,counts,k", [
    ("one lane's limit", [63, 64, 65, 0, 1, 8, 9, 7, 64, 200], 10),
    ("all long", [65] * 40, 7),
    ("all short", [1, 2, 3, 4, 5, 6] * 50, 300),
    ("mixed, chunked ranking", [1, 3, 0, 5, 2, 70, 4, 1] * 2500, 50),
    ("a tenth of the parents", [1, 2] * 5000, 1000),
])
def test_parent_lengths_match_oracle(rt, name, counts, k):
    from eos_amd.turboquant import TurboQuantIndex, TurboQuantParents
    print(f"[case] parents {name}", flush=True)
    off = _offsets(counts)
    n = int(off[-1])
    c = datagen.TurboQuantCorpus(n, 40, 2, 5, 6, 7)
    q = datagen.baseline_queries(3, 40, 8)
    idx = TurboQuantIndex(rt, c.codes, c.norms, c.dim, c.bits, c.codebook, c.codebook_scale,
                          c.rotation)
    par = TurboQuantParents(idx, off)
    for agg, top_n, pen in (("max", 1, 0.0), ("top2-mean", 2, 0.05), ("top5-mean", 5, 0.0)):
        got = par.top_k(q, k, agg, pen)
        want = oracle.tq_parent_topk(q, c.rotation, 40, 2, c.codebook, c.codebook_scale, c.codes,
                                     c.norms, off, k, top_n, pen)
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g, w)
    # a flat search after it: the shared candidate lists are reset
    ids, sc, _ = idx.top_k(q, min(5, n))
    wi, ws = oracle.tq_topk(q, c.rotation, 40, 2, c.codebook, c.codebook_scale, c.codes, c.norms,
                            min(5, n))
    np.testing.assert_array_equal(ids, wi)
    np.testing.assert_array_equal(sc, ws)
    par.release()
    idx.release()


@pytest.mark.parametrize("name,np_,nq,k", [
    ("split, eight lists of 1024 keys, the merge's limit", 77000, 2, 1024),
    ("split, seven lists above the smaller merge's limit", 76800, 2, 1025),
    ("split at 64 queries", 16500, 64, 40),
    ("just above the line", 24000, 3, 400),
    ("just below the line", 23999, 3, 400),
    ("large k on one workgroup a row", 33000, 2, 1000),
])
def test_parent_ranking_split(rt, name, np_, nq, k):
    """Parents' ranking split into chunks and not, at the edges of the merge."""
    from eos_amd.turboquant import TurboQuantIndex, TurboQuantParents
    print(f"[case] parent ranking: {name}", flush=True)
    off = np.arange(np_ + 1, dtype=np.int64)
    c = datagen.TurboQuantCorpus(np_, 24, 2, 15, 16, 17)
    norms = c.norms.copy()
    norms[np_ // 2:np_ // 2 + 40] = norms[0]  # more equal scores
    codes = c.codes.copy()
    codes[np_ // 2:np_ // 2 + 40] = codes[0]
    q = datagen.baseline_queries(nq, 24, 18)
    idx = TurboQuantIndex(rt, codes, norms, 24, 2, c.codebook, c.codebook_scale, c.rotation)
    par = TurboQuantParents(idx, off)
    got = par.top_k(q, k, "max", 0.0)
    want = oracle.tq_parent_topk(q, c.rotation, 24, 2, c.codebook, c.codebook_scale, codes, norms,
                                 off, k, 1, 0.0)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
    par.release()
    idx.release()
