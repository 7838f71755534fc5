"""Parents with children whose score is NaN (a query product that overflows
f32 times a Norm of zero): such a child counts as -infinity, by a lane (up to
64 children) as by a wavefront, wherever it lies among the others."""
import numpy as np
import pytest

from eos_amd import datagen

pytestmark = pytest.mark.gpu


def test_nan_child_scores_count_as_lowest(rt):
    from eos_amd.turboquant import TurboQuantIndex, TurboQuantParents
    print("[case] parents with NaN children", flush=True)
    counts = [1, 2, 3, 5, 8, 9, 40, 64, 65, 200] * 6
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    n = int(off[-1])
    c = datagen.TurboQuantCorpus(n, 32, 4, 31, 32, 33)
    # Products D alpha of standard deviation 1e38: a few per cent overflow.
    norms = np.where(np.arange(n) % 3 == 0, 0.0, 1e-3 * (1 + np.arange(n) % 17)).astype(np.float32)
    q = (datagen.baseline_queries(6, 32, 34).astype(np.float64) * 6e38).astype(np.float32)
    assert np.isfinite(q).all()
    idx = TurboQuantIndex(rt, c.codes, norms, 32, 4, c.codebook, c.codebook_scale, c.rotation,
                          zero_vector_allowed=True)
    _, scores = idx.inner_product_prepared(q)
    mixed = [any(np.isnan(scores[i, a:b]).any() and np.isfinite(scores[i, a:b]).sum() >= 1
                 for a, b in zip(off[:-1], off[1:])) for i in range(len(q))]
    assert any(mixed), "the case has no parent with NaN and finite children"
    par = TurboQuantParents(idx, off)
    for agg, top_n in (("max", 1), ("top2-mean", 2), ("top3-mean", 3), ("top5-mean", 5)):
        ids, got, _, _ = par.top_k(q, 0, agg)
        for i in range(len(q)):
            want = np.zeros(len(counts), np.float32)
            for p, (a, b) in enumerate(zip(off[:-1], off[1:])):
                ch = np.where(np.isnan(scores[i, a:b]), -np.inf, scores[i, a:b]).astype(np.float64)
                best = np.sort(ch)[::-1][:top_n]
                with np.errstate(all="ignore"):
                    want[p] = np.float32(sum(best.tolist()) / len(best))
            by_parent = np.zeros(len(counts), np.float32)
            by_parent[ids[i]] = got[i]
            np.testing.assert_array_equal(by_parent, want, err_msg=f"{agg} query {i}")
    par.release()
    idx.release()
