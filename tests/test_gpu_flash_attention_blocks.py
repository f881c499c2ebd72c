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


def _eight_waves(heads, seq):
    """The launcher's rule for 8-wave blocks at head_dim 128 (fwd_waves in
    flash_attn.hip), which has to change with it."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    blocks = heads * -(-seq // 256)
    return blocks % (2 * cus) == 0 or blocks >= 10 * cus


# two rounds of 256 blocks of 256 queries: 1, 2 and 4 blocks a head, their
# last ones full, one query, and ending inside a tile or a wave
@pytest.mark.parametrize("mode", ["softmax_native", "softcap_d4", "sigmoid_d3"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("heads,seq,valid", [(512, 1, -1), (512, 33, 32), (512, 250, 65), (512, 256, 129),
                                             (256, 257, -1), (256, 448, 385), (128, 1000, -1)])
def test_eight_wave_blocks_match_four(spline_ops, cuda, mode, causal, heads, seq, valid):
    print(f"blocks {mode} causal {causal} heads {heads} seq {seq} valid {valid}", flush=True)
    assert _eight_waves(heads, seq) and not _eight_waves(8, seq)
    q, k, v = (t.to(cuda) for t in _inputs(1, heads, heads // 8, seq, seq, d=128)[:3])
    got = _out(spline_ops, q, k, v, mode, causal, valid)
    few = _out(spline_ops, q[:, :, -8:], k[:, :, -1:], v[:, :, -1:], mode, causal, valid)
    assert torch.isfinite(got[0]).all()
    assert torch.equal(got[0][:, :, -8:], few[0])
    for a, b in zip(got[1:], few[1:]):
        assert torch.equal(a[:, -8:], b)


def _two_per_cu(batch, heads, seq):
    """The launcher's rule for causal softcap at head_dim 64 (fwd_spare_lds in
    flash_attn.hip), which has to change with it."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    each = heads * -(-seq // 128)
    return each >= cus and 2 * cus < batch * each <= 4 * cus


# grids of two to four blocks a CU run two blocks to a CU: two and a half, three
# and four, one batch element and several
@pytest.mark.parametrize("mode", ["softcap_native", "softcap_d4"])
@pytest.mark.parametrize("per_cu,batch,seq", [(0.5, 1, 513), (0.5, 1, 700), (0.5, 1, 1024), (0.25, 3, 500), (1, 4, 33)])
def test_softcap_grids_of_two_blocks_a_cu(spline_ops, cuda, mode, per_cu, batch, seq):
    heads = int(per_cu * torch.cuda.get_device_properties(0).multi_processor_count)
    print(f"two per CU {mode} batch {batch} heads {heads} seq {seq}", flush=True)
    assert _two_per_cu(batch, heads, seq) and not _two_per_cu(1, 8, seq)
    q, k, v = (t.to(cuda) for t in _inputs(batch, heads, heads // 8, seq, seq, qmul=4.0, d=64)[:3])
    got = _out(spline_ops, q, k, v, mode, True)
    few = _out(spline_ops, q[-1:, :, -8:], k[-1:, :, -1:], v[-1:, :, -1:], mode, True)
    assert torch.isfinite(got[0]).all()
    assert torch.equal(got[0][-1:, :, -8:], few[0]) and torch.equal(got[1][-1:, -8:], few[1])


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


@pytest.mark.parametrize("mode", ["softmax_d2", "softcap_native", "sigmoid_d4"])
@pytest.mark.parametrize("d,heads,seq", [(64, 6, 1), (64, 4, 200), (128, 4, 129), (128, 512, 33)])
def test_heads_first_output(spline_ops, cuda, mode, d, heads, seq):
    print(f"heads first {mode} d {d} heads {heads} seq {seq}", flush=True)
    assert d == 64 or _eight_waves(2 * heads, seq) == (heads == 512)  # batch 2
    q, k, v = (t.to(cuda) for t in _inputs(2, heads, heads // 2, seq, d + seq, d=d)[:3])
    args = (M[mode], 12, True, 1 / math.sqrt(d), 30.0, 0.0)
    out, lse = spline_ops.flash_attn_fwd_bf16(q, k, v, *args)
    first, kept, kept_lse = spline_ops.flash_attn_fwd_heads_first_bf16(q, k, v, *args, True)
    (alone,) = spline_ops.flash_attn_fwd_heads_first_bf16(q, k, v, *args, False)
    assert first.is_contiguous() and alone.is_contiguous()
    for a in (first, alone):
        assert torch.equal(a, out.transpose(1, 2))
    assert torch.equal(kept, out) and torch.equal(kept_lse, lse)


@pytest.mark.parametrize("heads,seq", [(4, 130), (1, 130), (1, 1)])
def test_misaligned_gradient_layouts(cuda, heads, seq):
    """A gradient whose transposed view is contiguous at an address or at
    strides that 16-byte loads cannot take is copied."""
    from sfu_repro.fa4 import FA4Config, build_fa4_module

    print(f"misaligned gradient heads {heads} seq {seq}", flush=True)
    module = build_fa4_module(FA4Config(), head_dim=64)
    q, k, v, do = (t.transpose(1, 2).contiguous().to(cuda) for t in _inputs(2, heads, heads, seq, 7, d=64))
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    out = module(*leaves)
    want = torch.autograd.grad(out, leaves, do, retain_graph=True)
    memory = torch.empty(do.numel() + 1, dtype=do.dtype, device=cuda)[1:]
    for shape in ((2, heads, seq, 64), (2, seq, heads, 64)):
        dout = memory.view(shape)
        dout = (dout if shape[1] == heads else dout.transpose(1, 2)).copy_(do)
        got = torch.autograd.grad(out, leaves, dout, retain_graph=True)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), shape


@pytest.mark.parametrize("own", [True, False])
def test_wrapper_output_and_gradient_layouts(cuda, own):
    """The module's output is contiguous and the caller's to edit, and the
    gradients are the same from a contiguous, a transposed, a misaligned and
    an expanded dout, by this package's kernels and by a runtime around them
    (whose calls keep the copies)."""
    from sfu_repro import fa4_runtime
    from sfu_repro.fa4 import FA4AttentionWrapper, FA4Config, resolve_fa4_config

    runtime = fa4_runtime.runtime()
    if not own:
        runtime["flash_attn_fwd"] = lambda *a, **kw: fa4_runtime.flash_attn_fwd(*a, **kw)
    module = FA4AttentionWrapper(resolve_fa4_config(FA4Config(), runtime=runtime), 64)
    q, k, v, do = (t.transpose(1, 2).contiguous().to(cuda) for t in _inputs(2, 4, 2, 130, 7, d=64))

    def grads(dout, edit=False):
        leaves = [t.clone().requires_grad_() for t in (q, k, v)]
        out = module(*leaves)
        assert out.is_contiguous() and out.shape == q.shape
        with torch.no_grad():
            assert torch.equal(module(q, k, v), out)
        if edit:
            out.mul_(2)
        return torch.autograd.grad(out, leaves, dout)

    shifted = torch.empty(do.numel() + 1, dtype=do.dtype, device=cuda)[1:].view_as(do).copy_(do)
    row = do[:1, :1].expand_as(do)
    want = grads(do)
    for name, got, ref in (("transposed", grads(do.transpose(1, 2).contiguous().transpose(1, 2)), want),
                           ("misaligned", grads(shifted), want),
                           ("expanded", grads(row), grads(row.contiguous())),
                           ("edited", grads(do / 2, edit=True), want)):  # halves and doubles are exact
        assert all(torch.equal(a, b) for a, b in zip(got, ref)), name


# rows past the last key reach the products with probability 0: they hold
# zeros, not a copy of a row whose infinity would make them NaN.  4- and
# 8-wave blocks, a tile's first, middle and last row
@pytest.mark.parametrize("mode", ["softmax_native", "softcap_native", "sigmoid_native"])
@pytest.mark.parametrize("d,heads,seq", [(64, 4, 65), (64, 4, 200), (128, 4, 127), (128, 512, 33)])
def test_infinite_last_row_of_v(spline_ops, cuda, mode, d, heads, seq):
    print(f"infinite v {mode} d {d} heads {heads} seq {seq}", flush=True)
    q, k, v = (t.to(cuda) for t in _inputs(1, heads, heads, seq, d + seq, d=d)[:3])
    assert d == 64 or _eight_waves(heads, seq) == (heads == 512)
    v[:, -1, :, 3] = float("inf")
    out = spline_ops.flash_attn_fwd_bf16(q, k, v, M[mode], 12, False, 1 / math.sqrt(d), 30.0, 0.0, -1)[0]
    assert (out[..., 3] == float("inf")).all()
    assert torch.isfinite(out[..., :3]).all() and torch.isfinite(out[..., 4:]).all()
