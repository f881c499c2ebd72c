"""The gradient that reaches this package's backward kernels through the
attention module: rows at 16-byte aligned addresses whatever storage the
caller's gradient has.  On the CPU, with the kernels replaced by recorders."""

import pytest
import torch

from sfu_repro import fa4_runtime
from sfu_repro.fa4 import FA4AttentionWrapper, FA4Config, resolve_fa4_config


def _at(offset, *shape):
    n = torch.Size(shape).numel()
    return torch.arange(n + offset, dtype=torch.float32).to(torch.bfloat16)[offset:].view(shape)


GRADIENTS = {
    "contiguous": lambda b, h, s, d: _at(0, b, h, s, d),
    "misaligned": lambda b, h, s, d: _at(1, b, h, s, d),
    "transposed": lambda b, h, s, d: _at(0, b, s, h, d).transpose(1, 2),
    "transposed and misaligned": lambda b, h, s, d: _at(3, b, s, h, d).transpose(1, 2),
    "expanded": lambda b, h, s, d: _at(1, 1, 1, 1, d).expand(b, h, s, d),
    # dimensions of size 1 are contiguous at any stride
    "odd strides": lambda b, h, s, d: _at(0, b, h, s, d).as_strided(
        (b, h, s, d), [h * s * d if b > 1 else 3, s * d if h > 1 else 5, d if s > 1 else 7, 1]),
}


@pytest.mark.parametrize("name", list(GRADIENTS))
@pytest.mark.parametrize("batch,heads,seq", [(2, 4, 5), (2, 1, 5), (1, 4, 1), (1, 1, 1)])
def test_rows_reach_the_kernels_aligned(monkeypatch, name, batch, heads, seq):
    seen = []

    def forward(q, k, v, *, keep, **kw):
        return q.transpose(1, 2).clone(), q.clone(), torch.zeros(batch, heads, seq)

    def backward(q, k, v, out, dout, lse, *args, **kw):
        seen.append(dout)
        return torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)

    monkeypatch.setattr(fa4_runtime, "flash_attn_fwd_heads_first", forward)
    monkeypatch.setattr(fa4_runtime, "flash_attn_bwd", backward)
    module = FA4AttentionWrapper(resolve_fa4_config(FA4Config(), runtime=fa4_runtime.runtime()), 64)
    q, k, v = (torch.zeros(batch, heads, seq, 64, dtype=torch.bfloat16, requires_grad=True) for _ in range(3))
    dout = GRADIENTS[name](batch, heads, seq, 64)
    module(q, k, v).backward(dout)
    (rows,) = seen
    assert torch.equal(rows, dout.transpose(1, 2))
    assert rows.data_ptr() % 16 == 0 and rows.stride(3) == 1 and all(n % 8 == 0 for n in rows.stride()[:3])
    if name == "contiguous":
        assert rows.data_ptr() == dout.data_ptr()  # read where it lies
