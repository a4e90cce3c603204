"""Static checks of the compiled GEMM kernels (CPU only, needs hipcc).

The 16x16x32 main loop names its accumulation registers (AGPRs) literally in
inline asm, so the compiler must never place a value of its own there.  It
does so only under register pressure (a copy `v_accvgpr_write_b32 aN, vM` and
back).  ccfuser_amd.build runs this scan on every build and refuses to link a
library that fails it; these tests run the same scan and also check that it
sees the kernels it is meant for.
"""
import shutil
from pathlib import Path

import pytest

needs_hipcc = pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(),
                                 reason="hipcc not available")


@needs_hipcc
def test_no_compiler_values_in_accumulation_registers(tmp_path):
    from ccfuser_amd import build as B
    text = B.device_assembly("ffn.hip", tmp_path / "ffn.s")
    kernels = B.kernel_bodies(text, B.ACC_CHECKED["ffn.hip"])
    # plain, persistent, split-tail kernels, each in several epilogue forms
    assert len(kernels) >= 10, [k for k, _ in kernels]
    assert any("persistent" in k for k, _ in kernels) and any("tail" in k for k, _ in kernels)
    for name, body in kernels:
        assert body.count("v_mfma_f32_16x16x32_f16") >= 128, name
        assert "s_endpgm" in body, name
    assert B.acc_register_violations(text, B.ACC_CHECKED["ffn.hip"]) == []


@needs_hipcc
def test_probe_kernel_keeps_the_accumulation_registers_to_itself(tmp_path):
    """The MFMA-only probe names all 256 accumulation registers in inline asm too: the compiler
    must hold nothing of its own there (a value parked in one would be overwritten: it was the
    index of the kernel's only store once), and must not spill."""
    from ccfuser_amd import build as B
    text = B.device_assembly("probe.hip", tmp_path / "probe.s")
    kernels = B.kernel_bodies(text, B.ACC_CHECKED["probe.hip"])
    assert len(kernels) == 1
    assert kernels[0][1].count("v_mfma_f32_16x16x32_f16") == 64
    assert B.acc_register_violations(text, B.ACC_CHECKED["probe.hip"]) == []


def test_the_scan_flags_a_parked_value_and_code_behind_an_early_exit():
    """The scan itself, on hand-made assembly: a compiler-style accumulation-register copy is
    found also when it sits behind the kernel's first s_endpgm."""
    from ccfuser_amd import build as B
    asm = """
_ZN3ccf12_GLOBAL__N_119grouped_gemm_kernelIXX:        ; @kernel
\ts_cbranch_scc1 .LBB0_2
\ts_endpgm
.LBB0_2:
\tv_mfma_f32_16x16x32_f16 a[0:3], v[0:3], v[4:7], a[0:3]
\tv_accvgpr_write_b32 a17, v3
\ts_endpgm
.Lfunc_end0:
_ZN3ccf5otherE:
\tv_accvgpr_write_b32 a1, v1
.Lfunc_end1:
"""
    bad = B.acc_register_violations(asm, B.ACC_CHECKED["ffn.hip"])
    assert len(bad) == 1 and "a17" in bad[0][1][0]
    clean = asm.replace("\tv_accvgpr_write_b32 a17, v3\n", "\tv_accvgpr_write_b32 a[17], 0\n")
    assert B.acc_register_violations(clean, B.ACC_CHECKED["ffn.hip"]) == []


@needs_hipcc
def test_gate_kernels_keep_their_values_in_registers(tmp_path):
    """Both forms of the fp16 gate (wavefronts sharing K, and every wavefront alone through all of K
    with four sets of loads in flight) are built for a register budget: none of their instantiations
    may spill (the kernel metadata's private segment size is what a spill would need)."""
    import re
    from ccfuser_amd import build as B
    text = B.device_assembly("gate.hip", tmp_path / "gate.s")
    sizes = {}
    for m in re.finditer(r"\.name:\s+(\S*gate_(?:mfma|stream)_kernel\S*)(.*?)\.private_segment_fixed_size:\s+(\d+)", text, flags=re.S):
        if ".name:" in m.group(2):                      # ran into the next kernel's record
            continue
        sizes[m.group(1)] = int(m.group(3))
    forms = {"mfma": 0, "stream": 0}
    for name, size in sizes.items():
        assert size == 0, f"{name} spills {size} bytes"
        forms["stream" if "stream" in name else "mfma"] += 1
    # tile widths 16 and 32, 1/2/4 slots, three list lengths of the selection
    assert forms["mfma"] >= 15 and forms["stream"] >= 15, forms


def _few_rows_kernels(text):
    from ccfuser_amd import build as B
    return B.kernel_bodies(text, B.READS_CHECKED["few.hip"])


@needs_hipcc
def test_few_row_kernels_touch_no_read_in_flight(tmp_path):
    """The few-row tiles read a half K step's fragments ahead of their use, in inline asm, across the loop's back edge: no
    instruction may name such a register before its wait, and nothing may spill.  With the waits for the older half left
    out, or one of its registers copied behind the reads, the scan finds it."""
    import re
    from ccfuser_amd import build as B
    text = B.device_assembly("few.hip", tmp_path / "few.s")
    kernels = _few_rows_kernels(text)
    assert len(kernels) == 10, [name for name, _ in kernels]
    spilled = B.spilled_bytes(text, B.READS_CHECKED["few.hip"])
    assert len(spilled) == 10 and not any(spilled.values()), spilled
    for name, body in kernels:
        assert body.count("ds_read_b128") >= 24, name
        assert B.pending_read_violations(body) == [], name
    body = kernels[-1][1]
    asm_waits = re.compile(r"(s_waitcnt lgkmcnt\()([1-9]\d*)(\))")
    assert len(asm_waits.findall(body)) >= 6                                # one per tile shape
    assert B.pending_read_violations(asm_waits.sub(lambda m: f"{m[1]}{int(m[2]) + 1}{m[3]}", body)) != []
    for read in list(re.finditer(r"\n\tds_read_b128 v\[(\d+):\d+\][^\n]*", body))[::40]:
        copy = f"\n\tv_mov_b32_e32 v255, v{read.group(1)}"
        assert B.pending_read_violations(body[:read.end()] + copy + body[read.end():]) != [], read.group(0)


@needs_hipcc
def test_256_row_kernels_copy_no_fragment_in_flight(tmp_path):
    """The 256-row tiles' main loop ends with the next tile's fragments being read.  The compiler copies them between the
    loops that it has for full and partly filled tiles, which must be behind their wait: a tile of few rows is through the
    rest of its last step before the reads are."""
    from ccfuser_amd import build as B
    text = B.device_assembly("ffn.hip", tmp_path / "ffn.s")
    kernels = [k for k in B.kernel_bodies(text, B.COPIES_CHECKED["ffn.hip"]) if "ds_read" in k[1]]
    assert len(kernels) >= 20, [name for name, _ in kernels]
    for name, body in kernels:
        assert B.pending_read_violations(body, copies_only=True) == [], name


@pytest.mark.parametrize("body,found", [
    # waited for, also where an older read is the one that is used
    ("ds_read_b128 v[0:3], v8\nds_read_b128 v[4:7], v8\ns_waitcnt lgkmcnt(1)\nv_mov_b32 v9, v0\ns_endpgm", []),
    ("ds_read_b128 v[0:3], v8\nds_read_b128 v[4:7], v8\ns_waitcnt lgkmcnt(1)\nv_mov_b32 v9, v4\ns_endpgm", ["v_mov_b32 v9, v4"]),
    # overwritten, and used as an address, while in flight
    ("ds_read_b32 v0, v8\nv_mov_b32 v0, 0\ns_waitcnt lgkmcnt(0)\ns_endpgm", ["v_mov_b32 v0, 0"]),
    ("ds_read_b32 v0, v8\nds_read_b32 v1, v0\ns_endpgm", ["ds_read_b32 v1, v0"]),
    # across a back edge: the second turn copies what the first one left in flight
    (".L1:\nv_mov_b32 v9, v1\nds_read_b32 v1, v8\ns_cbranch_scc1 .L1\ns_endpgm", ["v_mov_b32 v9, v1"]),
    (".L1:\nv_mov_b32 v9, v1\nds_read_b32 v1, v8\ns_waitcnt lgkmcnt(0)\ns_cbranch_scc1 .L1\ns_endpgm", []),
    # one of two ways to a place waits
    ("ds_read_b32 v1, v8\ns_cbranch_scc1 .L1\ns_waitcnt lgkmcnt(0)\n.L1:\nv_mov_b32 v9, v1\ns_endpgm", ["v_mov_b32 v9, v1"]),
    # memory loads have a count of their own; loads to LDS leave no register
    ("global_load_dword v1, v[8:9], off\ns_waitcnt lgkmcnt(0)\nv_mov_b32 v2, v1\ns_endpgm", ["v_mov_b32 v2, v1"]),
    ("global_load_dword v1, v[8:9], off\nglobal_load_lds_dwordx4 v[8:9], off\ns_waitcnt vmcnt(1)\nv_mov_b32 v2, v1\ns_endpgm", []),
    # a load behind another one to the same register comes back behind it
    ("ds_read_b32 v1, v8\nds_read_b32 v1, v7\ns_waitcnt lgkmcnt(0)\nv_mov_b32 v2, v1\ns_endpgm", []),
])
def test_the_scan_for_reads_in_flight(body, found):
    from ccfuser_amd import build as B
    assert B.pending_read_violations(body) == found


def test_the_scan_for_copies_only():
    from ccfuser_amd import build as B
    body = "ds_read_b32 v1, v8\nv_add_u32 v2, v1, v1\n{}\ns_waitcnt lgkmcnt(0)\nv_mov_b32 v3, v1\ns_endpgm"
    assert B.pending_read_violations(body.format("v_mov_b64 v[4:5], v[0:1]"), copies_only=True) == ["v_mov_b64 v[4:5], v[0:1]"]
    assert B.pending_read_violations(body.format("v_mov_b64 v[4:5], v[6:7]"), copies_only=True) == []


def test_the_scan_refuses_what_it_cannot_follow():
    from ccfuser_amd import build as B
    for line in ("s_swappc_b64 s[30:31], s[0:1]", "flat_load_dword v0, v[2:3]", "s_waitcnt 0x0"):
        with pytest.raises(ValueError):
            B.pending_read_violations(line + "\ns_endpgm")
