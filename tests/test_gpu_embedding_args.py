"""Embedding rows with the ids in the kernel's arguments (at most 512) and from
device memory (more), rows shorter and longer than a workgroup, bit for bit."""
import numpy as np
import pytest

import oracle
from runtimed_amd import rq, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", [rq.Q8_0, rq.Q4_0, rq.Q5_0, rq.Q4_K, rq.Q5_K, rq.Q6_K])
@pytest.mark.parametrize("n_ids", [1, 511, 512, 513])
@pytest.mark.parametrize("n,k", [(40, 128), (24, 1152)])
def test_rows(dev, qtype, n_ids, n, k):
    blocks = synth.weight_blocks(qtype, n + k, n, k)
    rc, wf = oracle.dequant_tensor(qtype, blocks, n * k)
    assert rc == 0
    ids = np.random.default_rng(n_ids).integers(0, n, n_ids).astype(np.uint32)
    ids[-1] = n - 1
    got = rq.QWeight(qtype, blocks, n, k).embedding(ids).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), wf.reshape(n, k)[ids].view(np.uint32))
