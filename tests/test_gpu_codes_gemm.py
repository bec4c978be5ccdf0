"""The codes GEMM (rq_cgemm.hip): prefill linears and Marlin products with the
integer codes on the f16 matrix cores, against the oracle's exact weights in
f64, where the kernel can go wrong: ragged rows and columns (a last column tile
that starts at n - 64), one pair of chunks and many, K split over waves and
workgroups, rows that start inside a block, an activation row of any magnitude,
infinities and NaN.

Bound per output: the activations keep 22 bits (2^-22 |x| each, none lost on
16-bit ones), sums of at most 64 products are added to the output's sum, so at
most 16 + k / 64 + 8 + 8 roundings of partial sums that are no larger than the
sum of |x| (|scaled code| + |min|), and the result is rounded to its type."""
import numpy as np
import pytest
import torch

import oracle
from runtimed_amd import rq, synth

pytestmark = pytest.mark.gpu

FORMATS = [rq.Q4_K, rq.Q5_K, rq.Q6_K, rq.Q8_0, rq.Q4_0, rq.Q5_0]
EPS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def weight(q, seed, n, k):
    blocks = synth.weight_blocks(q, seed, n, k)
    rc, w = oracle.dequant_tensor(q, blocks, n * k)
    assert rc == 0
    return rq.QWeight(q, blocks, n, k), w.reshape(n, k).astype(np.float64)


def spread(q, w):
    """|scaled code| + |min| of every weight, from above: the min of Q4_K / Q5_K is at most 63 dmin, dmin <= 1e-2."""
    return np.abs(w) + (2 * 0.63 if q in (rq.Q4_K, rq.Q5_K) else 0.0)


def check(y, x, w, mag, dtype, bias=None):
    xd = x.double().cpu().numpy()
    ref = xd @ w.T
    k = w.shape[1]
    bound = (2.0 ** -22 + (k / 64 + 32) * 2.0 ** -24) * (np.abs(xd) @ mag.T)
    if bias is not None:
        ref = ref + bias.double().cpu().numpy()
        bound = bound + 2 * EPS[dtype] * (np.abs(ref) + np.abs(bias.double().cpu().numpy()))
    bound = bound + EPS[dtype] * np.abs(ref) + 1e-30
    got = y.double().cpu().numpy()
    bad = np.abs(got - ref) > bound
    assert not bad.any(), (np.argwhere(bad)[:4], np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize("q", FORMATS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("m,n,k", [(65, 64, 1024), (130, 66, 1152), (97, 190, 2176), (65, 64, 8192)])
def test_one_weight(dev, q, dtype, m, n, k):
    w, wf = weight(q, 7 * n + k, n, k)
    x = torch.from_numpy(synth.activations(m + k, m, k)).to(dev).to(dtype)
    x *= torch.logspace(-3, 3, m, device=dev).to(dtype)[:, None] if dtype == torch.float32 else 1
    check(w.forward(x, out_dtype=torch.float32), x, wf, spread(q, wf), torch.float32)


@pytest.mark.parametrize("q", FORMATS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k", [(65, 128), (200, 896)])
def test_set_with_biases(dev, q, dtype, m, k):
    ns = [128, 64, 130]
    pairs = [weight(q, i + k, n, k) for i, n in enumerate(ns)]
    x = torch.from_numpy(synth.activations(m, m, k)).to(dev).to(dtype)
    biases = [torch.randn(ns[0], device=dev), None, torch.randn(ns[2], device=dev)]
    ys = rq.linear_multi([w for w, _ in pairs], x, biases, out_dtype=dtype)
    for y, (_, wf), b in zip(ys, pairs, biases):
        check(y, x, wf, spread(q, wf), dtype, b)


@pytest.mark.parametrize("q", FORMATS)
def test_extreme_rows(dev, q):
    """Rows of the largest, the smallest and no magnitude, infinities and NaN: the other rows are not
    touched, and a row with them has the products' own signs."""
    m, n, k = 70, 64, 1024
    w, wf = weight(q, 3, n, k)
    x = synth.activations(5, m, k)
    x[0] *= 1e30
    x[1] *= 1e-38
    x[2] = 0.0
    x[3, 17] = np.inf
    x[4, 200], x[4, 900] = np.inf, -np.inf
    x[5, 3] = np.nan
    x[6, 511] = -np.inf
    y = w.forward(torch.from_numpy(x).to(dev)).cpu().numpy().astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ wf.T
        for r in (3, 4, 5, 6):  # column by column: numpy's product may not follow IEEE on inf * 0
            ref[r] = [np.sum(x[r].astype(np.float64) * wf[c]) for c in range(n)]
    for r in (3, 4, 5, 6):
        assert np.array_equal(np.isnan(y[r]), np.isnan(ref[r])) and np.array_equal(
            y[r][~np.isnan(ref[r])], ref[r][~np.isnan(ref[r])]), r
    ok = [r for r in range(m) if r not in (3, 4, 5, 6)]
    xs = torch.from_numpy(x[ok])
    tiny = 2.0 ** -126 * k  # products below the normal range
    check(torch.from_numpy(y[ok]), xs, wf, spread(q, wf) + tiny / np.maximum(np.abs(x[1]).max(), 1e-45), torch.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(2, 16384, 2112), (65, 300, 4100), (64, 1040, 1056), (70, 64, 16001)])
def test_marlin(dev, dtype, m, n, k):
    assert m * n * k >= 67e6
    rng = np.random.default_rng(n + k)
    kc = (k + 31) // 32
    words = rng.integers(0, 2 ** 32, (kc, n, 4), dtype=np.uint64).astype(np.uint32)  # also past k
    s = rng.uniform(-0.02, 0.02, n).astype(np.float32)
    mw = rq.MarlinWeight(torch.from_numpy(words.view(np.int32)).to(dev), torch.from_numpy(s).to(dev), k, n)
    nib = (words[..., None] >> (4 * np.arange(8, dtype=np.uint32))) & 15  # [kc, n, 4, 8]
    wf = (nib.transpose(1, 0, 2, 3).reshape(n, kc * 32)[:, :k].astype(np.float64) - 8.0) * s[:, None].astype(np.float64)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dev).to(dtype)
    check(rq.marlin_gemv(x, mw), x, wf, np.abs(wf), dtype)
    if k % 8 == 0:  # an activation pointer that is not 16-byte aligned
        buf = torch.empty(m * k + 1, dtype=dtype, device=dev)
        xu = buf[1:].view(m, k)
        xu.copy_(x)
        check(rq.marlin_gemv(xu, mw), x, wf, np.abs(wf), dtype)


def test_graph_replays(dev):
    """Captured calls (packed activations and split sums in the stream's workspace) replay the eager bits."""
    m, n, k = 65, 64, 8192
    w, _ = weight(rq.Q4_K, 11, n, k)
    x = torch.from_numpy(synth.activations(9, m, k)).to(dev)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        out = torch.empty(m, n, device=dev)
        w.forward(x, out=out)
        st.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            w.forward(x, out=out)
        for i in range(3):
            x.mul_(1.5)
            eager = w.forward(x).clone()
            out.zero_()
            g.replay()
            st.synchronize()
            assert torch.equal(out, eager), i
