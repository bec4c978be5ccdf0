"""One decoded token through several long Q4_K weights in one launch: the same
bits as each weight alone, with odd row counts, biases and every activation
type, and sets that hold a weight the launch does not take."""
import pytest
import torch

from runtimed_amd import rq, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,k", [((4096, 4098), 2560), ((4100, 4096, 4128), 4096), ((4096, 4096), 8192),
                                  ((4096, 1024), 4096), ((4096, 4096), 2304)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("with_bias", [False, True])
def test_set_is_each_alone(dev, ns, k, dtype, with_bias):
    print(f"mx set ns={ns} k={k} {dtype}", flush=True)
    ws = [rq.QWeight(rq.Q4_K, synth.weight_blocks(rq.Q4_K, n + i, n, k), n, k) for i, n in enumerate(ns)]
    x = torch.from_numpy(synth.activations(k, 1, k)).to(dev).to(dtype)
    bs = [torch.randn(n, device=dev) for n in ns] if with_bias else None
    for i, y in enumerate(rq.linear_multi(ws, x, bs)):
        assert torch.equal(y, ws[i].forward(x, bias=bs[i] if with_bias else None))
