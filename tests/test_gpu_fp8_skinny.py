"""The FP8 product with K split over a workgroup's waves (few tiles, or k a
multiple of 16 but not of 128), against f64 on the same codes: one step of K and
fewer steps than waves, a step that ends inside K, row tiles of 16, 32 and 64
rows with a ragged last one, columns past n, and NaN codes, which stay in
their own row or column.

Bound per output: products of e4m3 values are exact in f16 products, a wave
adds at most k / 256 + 1 matrix products of 32 terms (at most 32 roundings each
counted once), eight waves are added, two scales multiplied."""
import numpy as np
import pytest
import torch

import oracle
from runtimed_amd import rq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 16), (1, 33, 128), (16, 64, 4096), (17, 31, 272), (33, 100, 2064),
                                   (65, 40, 144), (5, 4000, 4064), (129, 65, 1040), (200, 96, 32)])
@pytest.mark.parametrize("scaled", [True, False])
def test_against_f64(dev, m, n, k, scaled):
    print(f"fp8 m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m + n + k)
    xq = rng.integers(0, 256, (m, k), dtype=np.uint8)
    wq = rng.integers(0, 256, (n, k), dtype=np.uint8)
    xq[(xq & 0x7F) == 0x7F] = 0x3A
    wq[(wq & 0x7F) == 0x7F] = 0xB1
    lut = np.array([oracle.fp8_decode(c) for c in range(256)], np.float64)
    xs, ws = (rng.uniform(0.5, 2.0, c).astype(np.float32) if scaled else None for c in (m, n))
    put = lambda a: None if a is None else torch.from_numpy(a).to(dev)
    out = torch.empty((m, n), device=dev)
    rq.fp8_gemm_q(put(xq), put(xs), put(wq), put(ws), out)
    s = np.outer(xs, ws).astype(np.float64) if scaled else 1.0
    ref, mag = (lut[xq] @ lut[wq].T) * s, (np.abs(lut[xq]) @ np.abs(lut[wq]).T) * s
    assert np.all(np.abs(out.cpu().numpy() - ref) <= (k / 256 + 1 + 32 + 8 + 2) * 2.0 ** -24 * mag)
    # a NaN code reaches its row of x, or its row of w, and nothing else
    xq[m // 2, k - 1] = 0x7F
    wq[n // 2, 0] = 0xFF
    rq.fp8_gemm_q(put(xq), put(xs), put(wq), put(ws), out)
    nan = np.zeros((m, n), bool)
    nan[m // 2], nan[:, n // 2] = True, True
    assert np.array_equal(np.isnan(out.cpu().numpy()), nan)


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [256, 264, 512, 4096, 4104, 8224])
def test_rows_on_one_and_four_waves(dev, xdt, k):
    # a row of at most 64 16-byte chunks on one wave, longer ones on four
    x = (torch.randn(5, k, generator=torch.Generator().manual_seed(k)) * 3).to(xdt)
    x[1] = 0.0
    x[2, k - 1], x[3, 0], x[4, k // 2] = float("nan"), float("inf"), 60000.0
    xq, xs = rq.fp8_quantize(x.to(dev), rq.FP8_PER_TOKEN)
    want_q, want_s = oracle.fp8_quantize_rows(x.float().numpy())
    assert np.array_equal(xs.cpu().numpy().view(np.uint32), want_s.view(np.uint32))
    assert np.array_equal(xq.cpu().numpy(), want_q)
    xq, _ = rq.fp8_quantize(x.to(dev), rq.FP8_UNSCALED)
    assert np.array_equal(xq.cpu().numpy(), oracle.fp8_encode_array(x.float().numpy().reshape(-1)).reshape(5, k))
