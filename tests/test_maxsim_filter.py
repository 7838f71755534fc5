"""The MaxSim bound filter at its edges: 4 and 8 query groups a pass with odd
numbers of passes, short and long K, the largest sums its start value leaves
room for, and Norms across the float range. The filter only decides which
documents are scored, so its top-k equals the sort of the exhaustive scores,
bit for bit."""
import numpy as np
import pytest

from eos_amd import datagen


@pytest.mark.gpu
@pytest.mark.parametrize("bits,d,nq", [(2, 32, 8), (2, 128, 17), (4, 64, 5), (4, 128, 8),
                                       (2, 256, 3), (4, 256, 9), (2, 288, 5)])
def test_bound_filter_equals_exhaustive(rt, bits, d, nq):
    print(f"[case] maxsim filter bits={bits} d={d} nq={nq}", flush=True)
    from eos_amd.turboquant import TurboQuantIndex, TurboQuantMultiVectorIndex
    ndocs, doc_len, tokens = 16500, 32, 5
    c = datagen.TurboQuantCorpus(ndocs * doc_len, d, bits, 71, 72, 73)
    codes, norms = c.codes.copy(), c.norms.astype(np.float32).copy()
    q = datagen.unit_rows(datagen.normal(74, nq * tokens * d).reshape(-1, d)).reshape(nq, tokens, d)
    # Every coordinate of the rotated token at its largest, against rows of
    # the codebook's extreme levels: the largest |D_hi|.
    levels = np.asarray(c.codebook, np.float64)
    sign = np.where(np.arange(d) % 3 == 0, -1.0, 1.0)
    q[1, 0] = (sign / np.sqrt(d)) @ np.asarray(c.rotation, np.float64).reshape(d, d)
    code = np.where(sign > 0, int(np.argmax(levels)), int(np.argmin(levels)))
    per = 8 // bits
    row = np.zeros(codes.shape[1], np.uint8)
    for j in range(d):
        row[j // per] |= int(code[j]) << (bits * (j % per))
    for doc in (3, 16499):
        codes[doc * doc_len + 7] = row
    codes[11 * doc_len + 2] = ~row  # the complement of every level
    # Norms out of the fast bound's range, and tiny ones.
    norms[5 * doc_len:6 * doc_len] = 1e-38
    norms[9000 * doc_len + 31] = np.float32(2.0) ** 110
    norms[9001 * doc_len] = np.float32(2.0) ** 99
    q = q.astype(np.float32)
    idx = TurboQuantIndex(rt, codes, norms, d, bits, c.codebook, c.codebook_scale, c.rotation)
    mv = TurboQuantMultiVectorIndex(idx, doc_len)
    want = mv.scores(q, 0, ndocs)
    for k in (1, 90):
        ids, sc = mv.top_k(q, k)
        for i in range(nq):
            order = np.lexsort((np.arange(ndocs), -want[i]))[:k]
            np.testing.assert_array_equal(ids[i], order, err_msg=f"k={k} query {i}")
            np.testing.assert_array_equal(sc[i], want[i][order])
    idx.release()
