"""AMD ISA audit of the built library, the gfx950 counterpart of the
reference's SASS audit (autonumerics_zero/spline_ops/audit_sincos_sass.py
greps the disassembled CUDA kernels for MUFU opcodes to show that the
polynomial programs issue no hardware transcendental).  Here the gfx950 code
objects embedded in libspline_hip.so (this build's own output) are
disassembled with llvm-objdump and every kernel is classified by the program
its name carries:

* polynomial kernels issue no hardware transcendental: no v_exp, v_log,
  v_sin, v_cos, v_sqrt or v_rsq, and, in the kernel families that do no
  integer division, no v_rcp either (the compiler's 64-bit division
  expansion uses v_rcp_f32 on converted integers, as in the packed SwiGLU
  row / column split and the RoPE and attention index math);
* the hardware baselines, the hybrid kernels' transcendental lanes and the
  softmax attention issue theirs;
* no kernel issues packed FP32 arithmetic (v_pk_fma_f32, v_pk_mul_f32,
  v_pk_add_f32): the build turns the packed-fp32-ops target feature off;
* no kernel spills registers to scratch memory (the code objects' AMDGPU
  metadata), apart from one measured exception;
* every load from memory to LDS has its wait states: M0 written ahead of it,
  and five behind a vector instruction that wrote its scalar address.

Runs on the CPU (no GPU, no compute)."""

import collections
import os
import re
import struct
import subprocess
import tempfile

import pytest

import capi_helpers

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
OBJCOPY = "/opt/rocm/llvm/bin/llvm-objcopy"
BUNDLE_MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

HARD_TRANS = re.compile(r"^v_(exp|log|sin|cos|sqrt|rsq)_")
RCP = re.compile(r"^v_rcp_(f32|f16)")  # v_rcp_iflag_f32 (integer division) excluded
PACKED_F32 = re.compile(r"^v_pk_(fma|mul|add)_f32")


def _code_objects(lib_path: str, tmp: str) -> list:
    """gfx950 code objects of every offload bundle in the library's
    .hip_fatbin section (one bundle per translation unit)."""
    fatbin = os.path.join(tmp, "fatbin")
    subprocess.run([OBJCOPY, "--dump-section", f".hip_fatbin={fatbin}", lib_path, os.path.join(tmp, "stripped")],
                   check=True, capture_output=True)
    data = open(fatbin, "rb").read()
    objects = []
    for start in (m.start() for m in re.finditer(re.escape(BUNDLE_MAGIC), data)):
        (entries,) = struct.unpack_from("<Q", data, start + len(BUNDLE_MAGIC))
        p = start + len(BUNDLE_MAGIC) + 8
        for _ in range(entries):
            offset, size, triple_len = struct.unpack_from("<QQQ", data, p)
            p += 24
            triple = data[p:p + triple_len].decode()
            p += triple_len
            if triple.endswith("gfx950"):
                path = os.path.join(tmp, f"co{len(objects)}.o")
                with open(path, "wb") as f:
                    f.write(data[start + offset:start + offset + size])
                objects.append(path)
    return objects


READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def _kernel_metadata(obj: str) -> list:
    """(.name, .vgpr_spill_count, .private_segment_fixed_size) of every
    kernel in one code object's AMDGPU metadata note."""
    text = subprocess.run([READELF, "--notes", obj], check=True, capture_output=True, text=True).stdout
    records, cur = [], {}
    for line in text.splitlines():
        m = re.match(r"\s*(-\s+)?\.(\w+):\s+(.*)$", line)
        if not m:
            continue
        if m.group(1) and cur:  # a new list item starts a new kernel record
            records.append(cur)
            cur = {}
        cur[m.group(2)] = m.group(3).strip()
    if cur:
        records.append(cur)
    return [(r["name"], int(r.get("vgpr_spill_count", 0)), int(r.get("private_segment_fixed_size", 0)))
            for r in records if "name" in r and "vgpr_spill_count" in r]


@pytest.fixture(scope="module")
def metadata():
    if not os.path.exists(READELF) or not os.path.exists(OBJCOPY):
        pytest.skip("ROCm llvm-readelf / llvm-objcopy not found")
    assert os.path.exists(capi_helpers.LIB), "build the library first (__graft_entry__.build())"
    with tempfile.TemporaryDirectory() as tmp:
        rows = []
        for obj in _code_objects(capi_helpers.LIB, tmp):
            rows += _kernel_metadata(obj)
    demangled = subprocess.run(["c++filt"], input="\n".join(r[0] for r in rows), check=True,
                               capture_output=True, text=True).stdout.splitlines()
    return [(re.sub(r"\(.*", "", d), spill, scratch) for d, (_, spill, scratch) in zip(demangled, rows)]


LDS_LOAD = re.compile(r"^(global|buffer|scratch)_load_lds_|^buffer_load_\w+ .*\blds\b")
SGPRS = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\bvcc\b")
TWO_RESULTS = re.compile(r"^v_(\w*_co_\w+|div_scale_\w+|mad_[ui]64_\w+)$")  # a scalar one behind the vector one


def _sgprs(operands: str) -> set:
    out = set()
    for m in SGPRS.finditer(operands):
        if m.group(1):
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            out.add(int(m.group(3)) if m.group(3) else "vcc")
    return out


def _wait_state_faults(window: list, load: str) -> list:
    """What a load to LDS breaks, from the instructions ahead of it (nearest
    last; a branch target between them would only add wait states)."""
    address = _sgprs(load.split(None, 1)[1])
    faults, states, m0_seen = [], 0, False
    for line in reversed(window):
        op, _, rest = line.partition(" ")
        operands = rest.split(",")
        if states < 1 and operands[0].strip() == "m0":
            faults.append(f"M0 written {states} wait states ahead of: {load}")
        m0_seen = m0_seen or operands[0].strip() == "m0"
        if states < 5 and op.startswith("v_"):
            written = _sgprs(operands[0]) | (_sgprs(operands[1]) if TWO_RESULTS.match(op) else set())
            if written & address:
                faults.append(f"{line} {states} wait states ahead of: {load}")
        states += int(rest.split()[0]) + 1 if op == "s_nop" else 1
    return faults if m0_seen else faults + [f"no write of M0 ahead of: {load}"]


def test_wait_state_audit_counts():
    """The rules of _wait_state_faults on written-out sequences."""
    load = "global_load_lds_dwordx4 v6, s[34:35]"
    base, m0 = "v_readfirstlane_b32 s34, v1", "s_mov_b32 m0, s20"
    assert _wait_state_faults([base, m0, "s_nop 0"], load)
    assert _wait_state_faults([base, m0, "s_nop 2"], load)
    assert not _wait_state_faults([base, m0, "s_nop 3"], load)
    assert not _wait_state_faults(["v_readfirstlane_b32 s36, v1", m0, "s_nop 0"], load)
    assert _wait_state_faults(["v_add_co_u32_e64 v0, s[34:35], v1, v2", m0, "s_nop 0"], load)
    assert not _wait_state_faults(["v_add_f32_e32 v0, s34, v2", m0, "s_nop 0"], load)
    assert _wait_state_faults([m0], load) and _wait_state_faults(["s_nop 4"], load)


@pytest.fixture(scope="module")
def disassembly():
    """Demangled kernel name (without parameters) -> Counter of mnemonics, and
    -> [loads to LDS, the wait states that they lack, instructions that name
    M0]."""
    if not os.path.exists(OBJDUMP) or not os.path.exists(OBJCOPY):
        pytest.skip("ROCm llvm-objdump / llvm-objcopy not found")
    assert os.path.exists(capi_helpers.LIB), "build the library first (__graft_entry__.build())"
    out = collections.defaultdict(collections.Counter)
    lds_loads = collections.defaultdict(lambda: [0, [], 0])
    with tempfile.TemporaryDirectory() as tmp:
        objects = _code_objects(capi_helpers.LIB, tmp)
        assert objects, "no gfx950 code object in the library"
        for obj in objects:
            text = subprocess.run([OBJDUMP, "-d", "-C", "--no-show-raw-insn", "--no-leading-addr", obj],
                                  check=True, capture_output=True, text=True).stdout
            name, window = None, collections.deque(maxlen=8)
            for line in text.splitlines():
                m = re.match(r"^<(.+)>:$", line)
                if m:
                    name = re.sub(r"\(.*", "", m.group(1))
                    window.clear()
                    continue
                if name and line.startswith("\t"):
                    out[name][line.split()[0]] += 1
                    instruction = line.split("//")[0].strip()
                    if re.search(r"\bm0\b", instruction):
                        lds_loads[name][2] += 1
                    if LDS_LOAD.match(instruction):
                        lds_loads[name][0] += 1
                        lds_loads[name][1] += _wait_state_faults(list(window), instruction)
                    window.append(instruction)
    return out, lds_loads


@pytest.fixture(scope="module")
def kernels(disassembly):
    return disassembly[0]


def _uses(counter, pattern) -> list:
    return sorted(k for k in counter if pattern.match(k))


NATIVE_OR_HYBRID = re.compile(r"Native|Hybrid|exp2_(bf16|f32)_kernel<2,")
# families whose index math has no integer division
NO_DIVISION = re.compile(r"pt::(pairwise_kernel|pairwise_element_kernel|sincos_table_kernel|"
                         r"sincos_compute_kernel|sincos_f32_kernel|exp2_bf16_kernel|exp2_f32_kernel|b3_f32_kernel|"
                         r"ref_sincos_kernel)\b")
# sigmoid-attention modes with a score program: B3 (6), B3-D2 (7), BF16 D3-D6 (8-11)
POLY_ATTENTION = re.compile(r"pt::flash_(fwd|bwd_dkdv|bwd_dkdv256|bwd_dq)_kernel<(6|7|8|9|10|11),")


def _polynomial(name: str) -> bool:
    if NATIVE_OR_HYBRID.search(name):
        return False
    if POLY_ATTENTION.search(name):
        return True
    return bool(re.search(r"Prog<|Alg<|Softcap(Fwd|Bwd)\w*Op|B3\w*Op|B3D2|HalfTurn|Quarter|PairLut|"
                          r"RopeFixedPhase|RopeCachedTable|exp2_(bf16|f32)_kernel<([013-9]|1[0-2]),|b3_f32_kernel|ref_sincos_kernel",
                          name))


def test_audit_sees_every_family(kernels):
    assert len(kernels) > 900
    for family in ("pairwise_kernel", "packed_fwd_kernel", "sincos_compute_kernel", "rope_apply_kernel",
                   "flash_fwd_kernel", "flash_bwd_dkdv_kernel", "flash_bwd_dkdv256_kernel", "flash_bwd_dq_kernel",
                   "flash_bwd_dq_ds_kernel", "exp2_bf16_kernel"):
        assert any(f"pt::{family}<" in k for k in kernels), family
    poly = [k for k in kernels if _polynomial(k)]
    assert len(poly) > 500


def test_no_packed_fp32_arithmetic(kernels):
    bad = {k: _uses(c, PACKED_F32) for k, c in kernels.items() if _uses(c, PACKED_F32)}
    assert not bad, bad


def test_polynomial_kernels_issue_no_transcendental(kernels):
    bad = {}
    for name, counter in kernels.items():
        if not _polynomial(name):
            continue
        hits = _uses(counter, HARD_TRANS)
        if NO_DIVISION.search(name):
            hits += _uses(counter, RCP)
        if hits:
            bad[name] = hits
    assert not bad, bad


def test_loads_to_lds_have_their_wait_states(disassembly):
    """An SGPR written by a vector instruction (v_readfirstlane of an address,
    v_readlane of a spilled one) may be read as an address five wait states
    later, and M0 one wait state after it was written.  The compiler pads its
    own loads so; what inline assembly holds it does not see.  Nothing but
    these loads uses M0, which they overwrite."""
    _, lds_loads = disassembly
    for family in ("flash_fwd_kernel", "flash_bwd_dkdv256_kernel", "flash_bwd_dq_ds_kernel"):
        assert any(f"pt::{family}<" in k and n for k, (n, _, _) in lds_loads.items()), family
    bad = {k: faults[:2] for k, (_, faults, _) in lds_loads.items() if faults}
    assert not bad, (len(bad), list(bad.items())[:3])
    others = {k: (n, m0) for k, (n, _, m0) in lds_loads.items() if n and m0 != n}
    assert not others, list(others.items())[:3]


@pytest.mark.parametrize("pattern,needed", [
    (r"UnaryOp<pt::(F16|BF16)Native<", r"^v_exp_f32"),
    (r"pt::(NativeSinCos|F32Native|PairNative|RopeNativeAngle)\b", r"^v_(sin|cos)_f32"),
    (r"SoftcapNative\w*Op|B3NativeOp", r"^v_exp_f32"),
    (r"exp2_(bf16|f32)_kernel<2,", r"^v_exp_f32"),
    # the packed FP16 fractions run on packed FP16 arithmetic
    (r"exp2_(bf16|f32)_kernel<(5|10|12),", r"^v_pk_fma_f16"),
    (r"exp2_(bf16|f32)_kernel<7,", r"^v_pk_add_f16"),
    # the vector path (the element path is all polynomial: the transcendental
    # lanes exist only for whole 16-byte vectors)
    (r"pairwise_kernel<pt::Hybrid(Fwd|Bwd)Op", r"^v_exp_f32"),
    (r"pt::flash_fwd_kernel<0,", r"^v_exp_f32"),
])
def test_hardware_baselines_issue_their_transcendental(kernels, pattern, needed):
    matched = [k for k in kernels if re.search(pattern, k)]
    assert matched, pattern
    missing = [k for k in matched if not _uses(kernels[k], re.compile(needed))]
    assert not missing, missing


def test_no_register_spills_outside_the_measured_exception(metadata):
    """No kernel spills VGPRs to scratch memory, except the head_dim-64
    dK/dV kernels of the softmax modes, which are held to 128 VGPRs for four
    waves per SIMD and spill at most a few registers (measured faster than
    the unspilled two-wave form); their instantiations for sequences that are
    not a multiple of 128 (and the softcap D4 one) carry the row guards and
    spill up to 4 registers / 20 bytes.  No forward kernel spills, and none
    of the 256-key dK/dV and dS-reading dQ kernels.  The softcap dK/dV kernels at head_dim 64 that also store dS for the
    dS-keeping backward spill up to 10 registers / 28 bytes (measured: that
    backward is still 1.1-1.3x the recomputing one)."""
    assert len(metadata) > 900
    softmax = r"(0|1|2|1[2-9]|2[01])"  # modes with an exp2 program or the hardware exp2
    aligned = re.compile(rf"pt::flash_bwd_dkdv_kernel<{softmax}, 0, \d+, 64, 8, false, false>$")
    ragged = re.compile(rf"pt::flash_bwd_dkdv_kernel<{softmax}, 0, \d+, 64, 8, true, false>$|"
                        r"pt::flash_bwd_dkdv_kernel<4, \d, 0, 64, 8, true, false>$")
    keeps_ds = re.compile(r"pt::flash_bwd_dkdv_kernel<[34], \d, 0, 64, 8, false, true>$")
    forward = [n for n, spill, scratch in metadata if "flash_fwd_kernel<" in n and (spill or scratch)]
    assert not forward, forward
    bad = [(n, spill, scratch) for n, spill, scratch in metadata
           if (spill or scratch) and not (aligned.search(n) and spill <= 4 and scratch <= 16)
           and not (ragged.search(n) and spill <= 4 and scratch <= 20)
           and not (keeps_ds.search(n) and spill <= 10 and scratch <= 28)]
    assert not bad, bad
