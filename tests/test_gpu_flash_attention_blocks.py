"""Block shapes and staging of the attention forward: the same queries give
the same bits from 8-wave blocks (chosen where they fill whole rounds of the
CUs) as from 4-wave blocks, and from rows so far apart that a staging
address needs 64 bits as from contiguous ones.  The 4-wave blocks' results
are compared with the float32 reference by the mode matrix."""

import math

import pytest
import torch

from attention_reference import M
from test_gpu_flash_attention_bwd import _inputs

pytestmark = pytest.mark.gpu


def _out(ext, q, k, v, mode, causal, valid=-1):
    out, lse = ext.flash_attn_fwd_bf16(q, k, v, M[mode], 12, causal, 1 / math.sqrt(q.shape[3]), 30.0, 0.0, valid)
    return (out, lse) if lse.any() else (out,)


# one round of 512 blocks of 256 queries: 1, 2 and 4 blocks a head, their
# last ones full, one query, and ending inside a tile or a wave
@pytest.mark.parametrize("mode", ["softmax_native", "softcap_d4", "sigmoid_d3"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("heads,seq,valid", [(512, 1, -1), (512, 33, 32), (512, 250, 65), (512, 256, 129),
                                             (256, 257, -1), (256, 448, 385), (128, 1000, -1)])
def test_eight_wave_blocks_match_four(spline_ops, cuda, mode, causal, heads, seq, valid):
    print(f"blocks {mode} causal {causal} heads {heads} seq {seq} valid {valid}", flush=True)
    q, k, v = (t.to(cuda) for t in _inputs(1, heads, heads // 8, seq, seq, d=128)[:3])
    got = _out(spline_ops, q, k, v, mode, causal, valid)
    few = _out(spline_ops, q[:, :, -8:], k[:, :, -1:], v[:, :, -1:], mode, causal, valid)
    assert torch.isfinite(got[0]).all()
    assert torch.equal(got[0][:, :, -8:], few[0])
    for a, b in zip(got[1:], few[1:]):
        assert torch.equal(a[:, -8:], b)


@pytest.mark.parametrize("d", [64, 128])
def test_rows_past_32_bit_offsets(spline_ops, cuda, d):
    print(f"wide rows d {d}", flush=True)
    q, k, v = (t.to(cuda) for t in _inputs(1, 2, 2, 9, d, d=d)[:3])
    step = (1 << 27) + 8
    base = torch.empty(8 * step + 2 * d, dtype=torch.bfloat16, device=cuda)
    wide = base.as_strided((1, 9, 2, d), (9 * step, step, d, 1))
    want = _out(spline_ops, q, k, v, "softmax_native", True)
    for i, t in enumerate((q, k, v)):
        wide.copy_(t)
        got = _out(spline_ops, *(wide if j == i else s for j, s in enumerate((q, k, v))), "softmax_native", True)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), ("qkv"[i], d)
