"""MaxSim document lists: wavefronts that keep more than 64 documents' results
(so that they append more than once), lists that hold most of the corpus or
overflow, thresholds that cannot prune, and one to eight query groups a pass.
The lists only decide which documents are scored, so the top-k equals the sort
of the exhaustive scores, bit for bit."""
import numpy as np
import pytest

from eos_amd import datagen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,d,ndocs,nq,ks", [
    (2, 32, 70000, 32, (1, 512)),     # 8 groups a pass, 91 documents a wavefront
    (2, 32, 230001, 1, (1, 2, 512)),  # one pass of 4 groups, one live
    (4, 64, 16384, 9, (500,)),        # three passes, lists of most documents
    (2, 384, 33000, 5, (3, 300)),     # 2 groups a pass
    (2, 1024, 17000, 3, (1, 200)),    # one group a pass
])
def test_lists_equal_exhaustive(rt, bits, d, ndocs, nq, ks):
    print(f"[case] maxsim lists bits={bits} d={d} ndocs={ndocs} nq={nq}", flush=True)
    from eos_amd.turboquant import TurboQuantIndex, TurboQuantMultiVectorIndex
    tokens = 4
    c = datagen.TurboQuantCorpus(ndocs * 32, d, bits, 81, 82, 83)
    q = datagen.unit_rows(datagen.normal(84, nq * tokens * d).reshape(-1, d))
    q = q.reshape(nq, tokens, d).astype(np.float32)
    q[nq // 2] = 0  # every score 0: the threshold lists every document
    idx = TurboQuantIndex(rt, c.codes, c.norms, d, bits, c.codebook, c.codebook_scale, c.rotation)
    mv = TurboQuantMultiVectorIndex(idx, 32)
    want = mv.scores(q, 0, ndocs)
    for k in ks:
        ids, sc = mv.top_k(q, k)
        for i in range(nq):
            order = np.lexsort((np.arange(ndocs), -want[i]))[:k]
            np.testing.assert_array_equal(ids[i], order, err_msg=f"k={k} query {i}")
            np.testing.assert_array_equal(sc[i], want[i][order])
    idx.release()
