"""What the operators take as tensors and lists of tensors, and what they refuse, before any kernel runs (no GPU), and tensors that
are not plain ones (GPU)."""
import numpy as np
import pytest
import torch

import ms_custom_ops_amd as ops


def test_refused_without_a_gpu():
    x, w, s = torch.zeros((4, 64), dtype=torch.int8), torch.zeros((64, 32), dtype=torch.int8), torch.ones(32)
    for bad in (x, torch.nn.Parameter(s), s.t()):
        with pytest.raises(ValueError, match="take GPU tensors; got a tensor on cpu"):
            ops.quant_batch_matmul(bad, w, s)
    with pytest.raises(ValueError, match="take GPU tensors"):
        ops.grouped_matmul_v4_cops([x], [ops.as_qint4x2(w)], scale=[s], group_list=torch.zeros(1, dtype=torch.int64), split_item=3, group_type=0)
    for bad in (np.zeros((4, 64), np.int8), 3, "x", [x], object()):
        with pytest.raises(TypeError, match="expected a torch.Tensor, got " + type(bad).__name__):
            ops.quant_batch_matmul(bad, w, s)
    with pytest.raises(TypeError):
        ops.quant_batch_matmul(None, None, None)
    with pytest.raises(TypeError, match="expected a list of tensors"):
        ops.grouped_matmul_v4_cops(x, [w], scale=[s])
    with pytest.raises(TypeError):
        ops.grouped_matmul_v4_cops([None], [None])
    with pytest.raises(TypeError):
        ops.grouped_matmul_v4_cops(None, None)
    with pytest.raises(TypeError):
        ops.grouped_matmul_v4_cops(5, 5)


@pytest.mark.gpu
def test_views_subclasses_iterables_and_streams(device):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randint(-127, 128, (6, 64), generator=g, device="cuda", dtype=torch.int8)
    w = torch.randint(-127, 128, (64, 32), generator=g, device="cuda", dtype=torch.int8)
    s = torch.nn.Parameter(torch.rand(32, generator=g, device="cuda"))
    want = ((x[2:].cpu().double() @ w.cpu().double()).float().cuda() * s.detach()).half()   # (integer sums are exact)
    got = ops.quant_batch_matmul(x[2:], w, s)                                                  # a view with an offset, a Parameter
    assert type(got) is torch.Tensor and not got.requires_grad and torch.equal(got, want)
    assert torch.equal(ops.grouped_matmul_v4_cops((v for v in [x[2:]]), (w,), scale=iter([s]))[0].to(torch.float16), want)
    with pytest.raises(RuntimeError, match="not contiguous"):
        ops.quant_batch_matmul(x.t().contiguous().t(), w, s)
    with pytest.raises(TypeError, match="unsupported dtype torch.complex64"):
        ops.quant_batch_matmul(x.to(torch.complex64), w, s)
    with pytest.raises(torch.OutOfMemoryError):
        ops.quant_batch_matmul(x[:1].expand(1 << 46, 64), w, s)                                # the result alone is 4 PiB
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        on_side = ops.quant_batch_matmul(x[2:], w, s)
    side.synchronize()
    assert torch.equal(on_side, want)
