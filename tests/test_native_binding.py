"""The native binding takes the plain form of a call and leaves every other
one to the general path (None), on the CPU; on a GPU both give the same bits
and raise the same errors."""
import pytest
import torch

from runtimed_amd import rq, synth


class _Weight:
    n, _hv = 3, 0


def test_other_forms_are_left_to_the_general_path():
    n, x = rq._native(), torch.zeros(2, 3)
    w = _Weight()
    assert n.linear(w, x, None, None) is None
    assert n.linear(w, [1.0], None, None) is None
    assert n.linear_multi([w], x, None, None) is None
    assert n.linear_multi(iter([w]), x, None, None) is None
    assert n.fp8_gemm(x, x.to(torch.float8_e4m3fn), None, 1, torch.float32) is None
    assert n.marlin(x, x, x, 3, 3) is None
    assert n.kv_pair(x, x, 1, torch.uint8) is None
    assert n.kv_dequantize(x, x, 1, torch.float32) is None


@pytest.mark.gpu
def test_same_bits_and_errors(dev):
    k = 512
    ws = [rq.QWeight(rq.Q8_0, synth.weight_blocks(rq.Q8_0, i, n, k), n, k) for i, n in enumerate((96, 64))]
    x = torch.randn(2, 3, k, device=dev, dtype=torch.bfloat16)
    bias = torch.randn(96, device=dev)
    for out_dtype in (None, torch.float32, torch.float16):
        y = ws[0].forward(x, out_dtype, bias=bias)
        want = torch.empty(2, 3, 96, device=dev, dtype=out_dtype or x.dtype)
        ws[0].forward(x, out=want, bias=bias)
        assert y.dtype == want.dtype and torch.equal(y, want)
    # not contiguous: the general path makes the copy
    wide = torch.randn(3, 2, k, device=dev, dtype=torch.bfloat16)
    assert torch.equal(ws[0].forward(wide.transpose(0, 1)), ws[0].forward(wide.transpose(0, 1).contiguous()))
    outs = rq.linear_multi(ws, x, [bias, None])
    want = [torch.empty_like(o) for o in outs]
    rq.linear_multi_into(ws, x, want, [bias, None])
    assert all(torch.equal(a, b) for a, b in zip(outs, want))
    # on a stream of its own, the output belongs to that stream
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y = ws[1].forward(x)
    s.synchronize()
    assert torch.equal(y, ws[1].forward(x))
    with pytest.raises(rq.RqError) as e:
        ws[0].forward(x[..., :32].contiguous())
    assert e.value.kind == "Shape" and "expected last dim 512, got 32" in str(e.value)
    with pytest.raises(TypeError):
        ws[0].forward(x.double())
    ws[0].close()
    with pytest.raises(rq.RqError) as e:
        ws[0].forward(x)
    assert e.value.kind == "Arg"
    # vmap: no raw pointer of a batch wrapper is taken
    with pytest.raises(Exception):
        torch.vmap(ws[1].forward)(x)
