"""The codes GEMM on at most 64 rows of x: tiles of 32 rows (m <= 32) and of 64,
on both sides of the rules that choose it, K split over waves and workgroups,
a ragged last column tile, sets with biases, rows with infinities and NaN.

Bound per output as for many rows (22 bits of x, at most 16 + k / 64 + 8 + 8
roundings of partial sums), or that of the small-M kernels where they run: x
as two bf16 limbs (2^-16)."""
import pytest
import torch

import oracle
from runtimed_amd import rq, synth

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def weight(q, seed, n, k, dev):
    blocks = synth.weight_blocks(q, seed, n, k)
    rc, w = oracle.dequant_tensor(q, blocks, n * k)
    assert rc == 0
    return rq.QWeight(q, blocks, n, k), torch.from_numpy(w.reshape(n, k)).to(dev).double()


def check(y, x, w, q, bias=None):
    xd, k = x.double(), w.shape[1]
    mag = w.abs() + (2 * 0.63 if q in (rq.Q4_K, rq.Q5_K) else 0.0)  # min at most 63 dmin, dmin <= 1e-2
    ref = xd @ w.t()
    bound = (2.0 ** -16 + (k / 64 + 32) * 2.0 ** -24) * (xd.abs() @ mag.t())
    if x.dtype == torch.bfloat16:  # the small-M kernel rounds the weights to bf16
        bound = bound + 2.0 ** -8 * (xd.abs() @ w.abs().t())
    if bias is not None:
        ref = ref + bias.double()
        bound = bound + 2 * EPS[y.dtype] * (ref.abs() + bias.double().abs())
    bound = bound + EPS[y.dtype] * ref.abs() + 1e-30
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("q", [rq.Q4_K, rq.Q5_K, rq.Q6_K, rq.Q8_0, rq.Q4_0, rq.Q5_0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_rows_on_a_long_weight(dev, q, dtype):
    n, k = 2050, 8192
    wt, w = weight(q, 5, n, k, dev)
    for m in (3, 4, 16, 17, 31, 32, 33, 64):
        print(f"codes q={q} {dtype} m={m}", flush=True)
        x = torch.from_numpy(synth.activations(m, m, k)).to(dev).to(dtype)
        check(wt.forward(x), x, w, q)


@pytest.mark.parametrize("q", [rq.Q4_K, rq.Q6_K, rq.Q8_0])
@pytest.mark.parametrize("m,ns,k", [(2, (13000, 70), 4096), (3, (8000, 8400), 2048), (5, (8000, 8400), 2048),
                                    (24, (2048, 2114), 2048), (24, (1024, 2114), 2048), (40, (2048, 2114), 2048)])
def test_sets_with_biases(dev, q, m, ns, k):
    print(f"codes set q={q} m={m} ns={ns} k={k}", flush=True)
    pairs = [weight(q, n, n, k, dev) for n in ns]
    x = torch.from_numpy(synth.activations(m + k, m, k)).to(dev)
    b = [torch.randn(n, device=dev) for n in ns]
    for y, (_, w), bias in zip(rq.linear_multi([p[0] for p in pairs], x, b), pairs, b):
        check(y, x, w, q, bias)


def test_rows_that_are_not_finite(dev):
    n, k, m = 2050, 8192, 7
    wt, w = weight(rq.Q4_K, 9, n, k, dev)
    x = torch.from_numpy(synth.activations(1, m, k)).to(dev)
    x[2, 5], x[4, 9] = float("inf"), float("nan")
    y = wt.forward(x)
    ok = [0, 1, 3, 5, 6]
    check(y[ok], x[ok], w, rq.Q4_K)
    want = x[2].double() @ w.t()
    assert torch.equal(torch.isnan(y[2]), torch.isnan(want))
    inf = torch.isinf(want)
    assert bool(inf.any()) and torch.equal(y[2].double()[inf], want[inf])
    assert bool(torch.isnan(y[4]).all())


@pytest.mark.parametrize("m", [24, 70, 200])
@pytest.mark.parametrize("order", [(rq.Q8_0, rq.Q4_K, rq.Q6_K), (rq.Q4_K, rq.Q4_K, rq.Q6_K, rq.Q5_K)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_formats_that_share_a_pack(dev, m, order, dtype):
    # runs of several formats on one x, with the sums the K formats need and without
    k = 4096
    ws = [rq.QWeight(q, synth.weight_blocks(q, i, 2050, k), 2050, k) for i, q in enumerate(order)]
    x = torch.from_numpy(synth.activations(m, m, k)).to(dev).to(dtype)
    for w, y in zip(ws, rq.linear_multi(ws, x)):
        mag = w.dequantize().double().abs()
        ref = x.double() @ w.dequantize().double().t()
        tol = (2.0 ** -15 + EPS[dtype]) * (x.double().abs() @ (mag + (1.26 if w.qtype in (rq.Q4_K, rq.Q5_K) else 0)).t())
        assert bool(((y.double() - ref).abs() <= tol).all())
