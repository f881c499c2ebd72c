"""dK / dV in 256-key blocks (grids that fill the CUs at head_dim 128)
against the 128- and 64-key blocks that a few of the same heads run in: dS
is the same to the bit (so is dQ), and the FP32 sums over queries differ in
order only.  The small grids' results are compared with the float32
reference by the other backward tests."""

import math

import pytest
import torch

from attention_reference import M
from test_gpu_flash_attention_bwd import _inputs

pytestmark = pytest.mark.gpu


def _grads(ext, t, mode, grad, causal, route):
    q, k, v, do = t
    args = (causal, 1 / math.sqrt(128), 30.0, -math.log(q.shape[1]))
    out, lse = ext.flash_attn_fwd_bf16(q, k, v, M[mode], 12, *args, -1)
    return ext.flash_attn_bwd_bf16(q, k, v, out, do, lse, M[mode], grad, route, *args)


def _agree(got, want):
    """BF16 roundings of two FP32 sums of the same n terms, n <= 1000: one
    step of BF16 apart, or n 2^-24 of the terms' sum near zero (here below
    2^-12 of the largest result)."""
    a, b = got.float(), want.float()
    return bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -12 * b.abs().max()).all())


def _wide(heads, seq, causal):
    """The launcher's rule for 256-key blocks at head_dim 128
    (dkdv_wide_blocks in flash_attn_bwd.hip), which has to change with it."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    blocks = heads * -(-seq // 256)
    if causal:
        return blocks >= 2 * cus
    return 19 * -(-blocks // cus) <= 10 * -(-heads * -(-seq // 128) // cus)


# two rounds of 256-key blocks under the mask; without it one round where
# 128-key blocks take two, or two where they take four (heads per CU).  One key
# and one wave's keys (without the mask so few never take these blocks), the
# block's middle and end, one key into its second half and into the second
# block, dS kept (256, 384, 512) or not
@pytest.mark.parametrize("mode,grad,route", [("softmax_native", 0, 0), ("softmax_d2", 0, 32), ("softmax_d2", 0, 14),
                                             ("softcap_d4", 1, 0), ("sigmoid_d3", 0, 0)])
@pytest.mark.parametrize("causal,per_cu,group,seq", [
    (True, 2, 4, 1), (True, 2, 1, 32), (True, 2, 4, 161), (True, 2, 1, 256), (True, 1, 8, 257), (True, 1, 4, 384),
    (True, 0.5, 4, 1000),
    (False, 1, 4, 129), (False, 1, 1, 161), (False, 1, 8, 256), (False, 0.5, 4, 257), (False, 0.5, 1, 384),
    (False, 1, 4, 385), (False, 1, 4, 512), (False, 0.25, 4, 1000)])
def test_wide_blocks_match_narrow(spline_ops, cuda, mode, grad, route, causal, per_cu, group, seq):
    heads = int(per_cu * torch.cuda.get_device_properties(0).multi_processor_count)
    print(f"dkdv {mode} route {route} causal {causal} heads {heads} group {group} seq {seq}", flush=True)
    assert _wide(heads, seq, causal) and not _wide(8, seq, causal)
    t = [x.to(cuda) for x in _inputs(1, heads, heads // group, seq, seq + group)]
    many = _grads(spline_ops, t, mode, grad, causal, route)
    few = _grads(spline_ops, [t[0][:, :, -8:], t[1][:, :, -8 // group:], t[2][:, :, -8 // group:], t[3][:, :, -8:]],
                 mode, grad, causal, route)
    assert all(torch.isfinite(g).all() for g in many)
    assert torch.equal(many[0][:, :, -8:], few[0])
    for a, b in zip(many[1:], few[1:]):
        assert _agree(a[:, :, -8 // group:], b)


def test_wide_blocks_rows_past_32_bit_offsets(spline_ops, cuda):
    print("dkdv wide rows", flush=True)
    assert _wide(512, 9, True)
    t = [x.to(cuda) for x in _inputs(1, 512, 512, 9, 5)]
    want = _grads(spline_ops, t, "softmax_native", 0, True, 0)
    step = (1 << 27) + 8
    base = torch.empty(8 * step + 512 * 128, dtype=torch.bfloat16, device=cuda)
    wide = base.as_strided((1, 9, 512, 128), (9 * step, step, 128, 1))
    for i in range(4):
        wide.copy_(t[i])
        got = _grads(spline_ops, [wide if j == i else x for j, x in enumerate(t)], "softmax_native", 0, True, 0)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), "q k v dout".split()[i]


# dQ from the kept dS: heads in eighths (mapped by XCD) or not, one tile to
# several rings of them
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("heads,group,seq", [(2, 1, 128), (8, 4, 256), (12, 4, 384), (24, 3, 128), (16, 2, 640)])
def test_dq_from_ds_matches_recomputed(spline_ops, cuda, monkeypatch, d, causal, heads, group, seq):
    print(f"dq d {d} causal {causal} heads {heads} group {group} seq {seq}", flush=True)
    q, k, v, do = (x.to(cuda) for x in _inputs(2, heads, heads // group, seq, seq + d, qmul=6.0, d=d))
    args = (causal, 1 / math.sqrt(d), 30.0, 0.0)
    out, lse = spline_ops.flash_attn_fwd_bf16(q, k, v, M["softcap_d4"], 4, *args, -1)
    got = spline_ops.flash_attn_bwd_bf16(q, k, v, out, do, lse, M["softcap_d4"], 1, 0, *args)
    monkeypatch.setenv("SPLINE_ATTN_DS_MAX_BYTES", "0")
    want = spline_ops.flash_attn_bwd_bf16(q, k, v, out, do, lse, M["softcap_d4"], 1, 0, *args)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("mode", ["softmax_native", "sigmoid_native"])
@pytest.mark.parametrize("heads", [512, 8])  # 256-key blocks, and smaller ones
def test_infinite_last_row_of_dout(spline_ops, cuda, mode, heads):
    """Queries past the sequence add zeros to dV, not a masked probability
    times the last row's infinity."""
    print(f"infinite dout {mode} heads {heads}", flush=True)
    assert _wide(heads, 161, False) == (heads == 512)
    t = [x.to(cuda) for x in _inputs(1, heads, heads, 161, 161)]
    t[3][:, -1, :, 3] = float("inf")
    dv = _grads(spline_ops, t, mode, 0, False, 0)[2]
    assert (dv[..., 3] == float("inf")).all()
    assert torch.isfinite(dv[..., :3]).all() and torch.isfinite(dv[..., 4:]).all()
