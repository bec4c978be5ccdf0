"""K / V pairs in one launch and the division-free encoder, bit-exact against
the oracle: values on, just below and just above every code boundary of a
head's scale, heads with an infinity (whose scale is infinite) or a NaN, chunks
shorter and longer than a workgroup's 4096 elements, rows of 4 and of 8."""
import numpy as np
import pytest
import torch

import oracle
from runtimed_amd import rq

pytestmark = pytest.mark.gpu


def kv(shape, seed):
    rng = np.random.default_rng(seed)
    t = (rng.standard_normal(shape) * rng.uniform(0.01, 20.0)).astype(np.float32)
    h, flat = shape[1], t.transpose(1, 0, 2, 3).reshape(shape[1], -1).copy()
    for i in range(h):
        top = np.abs(flat[i]).max()
        for top_code, ties in ((448.0, np.concatenate([np.arange(0.5, 8) / 512,  # e4m3 boundaries
                                                       *[(1 + np.arange(0.5, 8) / 8) * 2.0 ** e for e in range(-6, 9)]])),
                               (127.0, np.arange(0.5, 127))):
            sc = np.float32(max(np.float32(top) / np.float32(top_code), np.float32(1e-8)))
            at = (ties[ties < top_code].astype(np.float32) * sc).astype(np.float32)
            near = np.concatenate([np.nextafter(at, np.float32(-np.inf)), at, np.nextafter(at, np.float32(np.inf)), -at])
            pick = rng.choice(near, size=min(near.size, flat.shape[1] // 3), replace=False)
            flat[i, rng.choice(flat.shape[1] - 1, size=pick.size, replace=False) + 1] = pick
        flat[i, 0] = top
    if h > 1:
        flat[1, 1], flat[1, 2] = np.inf, np.nan
    t = flat.reshape(h, shape[0], *shape[2:]).transpose(1, 0, 2, 3)
    return torch.from_numpy(np.ascontiguousarray(t))


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 3, 16, 80), (2, 2, 37, 36), (1, 2, 97, 128), (1, 1, 5, 4)])
def test_pair_bit_exact(dev, int8, dtype, shape):
    k, v = kv(shape, 1).to(dtype), kv(shape, 2).to(dtype)
    mode = rq.KV_INT8 if int8 else rq.KV_FP8
    kq, vq, ks, vs, got_mode = rq.quantize_block_kv(16, k.to(dev), v.to(dev), mode)
    assert got_mode == mode
    for t, q, s in ((k, kq, ks), (v, vq, vs)):
        want_q, want_s = oracle.kv_quantize(t.float().numpy(), int8)
        assert np.array_equal(s.cpu().numpy().reshape(-1).view(np.uint32), want_s.view(np.uint32))
        assert np.array_equal(q.cpu().view(torch.uint8).numpy(), want_q)
        for dt in (torch.float32, torch.bfloat16, torch.float16):
            want = torch.from_numpy(oracle.kv_dequantize(want_q, want_s, int8)).to(dt)
            got = rq.dequantize_block(q, s, mode, dt).cpu()
            nan = torch.isnan(want)
            assert torch.equal(torch.isnan(got), nan)
            assert torch.equal(got[~nan], want[~nan])


def test_unlike_shapes_and_types(dev):
    k, v = kv((1, 2, 24, 64), 3), kv((1, 2, 40, 64), 4).to(torch.bfloat16)
    kq, vq, ks, vs, _ = rq.quantize_block_kv(16, k.to(dev), v.to(dev), rq.KV_FP8)
    for t, q, s in ((k, kq, ks), (v, vq, vs)):
        want_q, want_s = oracle.kv_quantize(t.float().numpy(), False)
        assert np.array_equal(q.cpu().view(torch.uint8).numpy(), want_q)
        assert np.array_equal(s.cpu().numpy().reshape(-1), want_s)
