"""Decode GEMVs on rows of more than 64 pieces (32 elements, 64 for Q6_K) and
many rows: the team layout on both sides of its rule (two-run formats with at
most 128 pieces a row and at least 7168 rows walk a row on one wave), with odd
row counts that leave workgroups of unequal length.

Bound per output: f32 activations and exact f32 weights, sums of at most 64
products a lane, then a tree: (64 + 16) roundings of partial sums that are no
larger than the sum of |x| (|scaled code| + |min|)."""
import numpy as np
import pytest
import torch

import oracle
from runtimed_amd import rq, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [rq.Q4_K, rq.Q5_K, rq.Q6_K, rq.Q8_0, rq.Q4_0, rq.Q5_0])
@pytest.mark.parametrize("n,k", [(4098, 4224), (7168, 2176), (8194, 2176), (4097, 4096), (4102, 8320), (4096, 16384)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_rows_many_rows(dev, q, n, k, dtype):
    print(f"gemv q={q} n={n} k={k} {dtype}", flush=True)
    blocks = synth.weight_blocks(q, n + k, n, k)
    rc, w = oracle.dequant_tensor(q, blocks, n * k)
    assert rc == 0
    w = torch.from_numpy(w.reshape(n, k)).to(dev).double()
    x = torch.from_numpy(synth.activations(k, 1, k)).to(dev).to(dtype)
    y = rq.QWeight(q, blocks, n, k).forward(x, out_dtype=torch.float32).double()
    xd = x.double()
    mag = w.abs() + (2 * 0.63 if q in (rq.Q4_K, rq.Q5_K) else 0.0)  # min at most 63 dmin, dmin <= 1e-2
    bound = 80 * 2.0 ** -24 * (xd.abs() @ mag.t())
    if q == rq.Q4_K and k % 512 == 0:  # the matrix cores: x as two bf16 limbs, 2^-17 of each
        bound = bound + 2.0 ** -17 * (xd.abs() @ mag.t())
    assert bool(((y - xd @ w.t()).abs() <= bound).all())
