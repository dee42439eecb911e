"""The one-pass gradient walk of clip_grad_norm_ (_hoststep.clip_scan,
grads_are) against the Python checks it stands in for: it takes exactly the
lists they take, and leaves the rest to them."""
import numpy as np
import pytest
import torch

import adana_amd
from adana_amd import _hoststep, clip


class _Sub(torch.Tensor):
    pass


def _params(grads):
    out = []
    for g in grads:
        p = torch.nn.Parameter(torch.zeros(0) if g is None else torch.zeros(g.shape, dtype=g.dtype, device=g.device))
        p.grad = g
        out.append(p)
    return out


def test_lists_left_to_the_python_checks():
    p, q = torch.nn.Parameter(torch.zeros(3)), torch.nn.Parameter(torch.zeros(2))
    grads, numels, ptrs, _, bf16 = _hoststep.clip_scan([p, q])        # no gradients
    assert (grads, numels, ptrs, bf16) == ([], b"", b"", False)
    p.grad = torch.ones(3)
    assert _hoststep.clip_scan([p, q]) is None                        # not on a GPU
    assert _hoststep.clip_scan([p, object()]) is None
    assert _hoststep.clip_scan([torch.zeros(2).as_subclass(_Sub)]) is None
    assert _hoststep.grads_are([p, q], [p.grad]) and not _hoststep.grads_are([p, q], [])
    assert not _hoststep.grads_are([p, q], [p.grad, p.grad]) and not _hoststep.grads_are([p, q], [p.grad.clone()])
    assert not _hoststep.grads_are([object()], []) and _hoststep.grads_are([q], [])


def _forms(dev):
    a = torch.arange(24.0, device=dev)
    yield "contiguous", a.view(4, 6), True
    yield "transposed", a.view(4, 6).t(), True
    yield "permuted", a.view(2, 3, 4).permute(2, 0, 1), True
    yield "channels last", torch.ones(2, 3, 4, 5, device=dev).contiguous(memory_format=torch.channels_last), True
    yield "offset view", a[1:], True
    yield "one value, odd stride", a.as_strided((1, 1), (7, 3)), True
    yield "size-1 dimension, odd stride", a.as_strided((4, 1, 6), (6, 99, 1)), True
    yield "0-d", a[3], True
    yield "empty", a[:0].view(0, 5), True
    yield "empty, odd strides", a.as_strided((3, 0), (17, 2)), True
    yield "columns with gaps", a.view(4, 6)[:, :4], False
    yield "every second", a[::2], False
    yield "expanded", a[:1].expand(5), False
    yield "overlapping windows", a.as_strided((4, 3), (1, 1)), False
    yield "float64", a.double(), False
    yield "float16", a.half(), False
    yield "sparse", a.view(4, 6).to_sparse(), False


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
def test_takes_what_the_python_checks_take():
    dev = "cuda:0"
    for dtype in (torch.float32, torch.bfloat16):
        for name, g, fits in _forms(dev):
            if g.dtype == torch.float32 and not g.is_sparse:
                # the same layout in this dtype (a clone may not keep it)
                base = torch.arange(200, dtype=dtype, device=dev)
                g = base.as_strided(g.shape, g.stride())
            other = torch.ones(3, dtype=dtype, device=dev)
            for grads in ([g, None, other], [other, g]):
                params = _params(grads)
                want = [x for x in grads if x is not None]
                try:
                    clip._validate(want)
                    general = True
                except (NotImplementedError, RuntimeError):
                    general = False
                found = _hoststep.clip_scan(params)
                assert general == fits == (found is not None), (name, dtype)
                if found is None:
                    with pytest.raises((NotImplementedError, RuntimeError)):
                        adana_amd.clip_grad_norm_(params, 1.0)
                    continue
                got, numels, ptrs, index, bf16 = found
                assert len(got) == len(want) and all(x is p.grad for x, p in zip(got, [p for p in params if p.grad is not None]))
                assert np.frombuffer(numels, np.int64).tolist() == [x.numel() for x in want]
                assert np.frombuffer(ptrs, np.uint64).tolist() == [x.data_ptr() for x in want]
                assert (index, bf16) == (0, dtype == torch.bfloat16)
    mixed = _params([torch.ones(3, device=dev), torch.ones(3, device=dev, dtype=torch.bfloat16)])
    cpu = _params([torch.ones(3, device=dev), torch.ones(3)])
    sub = _params([torch.ones(3, device=dev)])
    sub.append(torch.ones(2, device=dev).as_subclass(_Sub))
    assert all(_hoststep.clip_scan(x) is None for x in (mixed, cpu, sub))
