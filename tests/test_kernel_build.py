"""Register and LDS budgets of the bf16 attention kernels, read from the compiler's kernel metadata
(device-only assembly of kernels_attn.hip with the library's flags; no GPU needed).

The two-wave kernel (64-query tiles) must fit three waves per SIMD (<= 168 VGPRs) without spills,
and the four-wave kernel (128-query tiles, global layers) four waves per SIMD (<= 128 VGPRs), where
it keeps one spilled register outside its key loops.  Both use 24 KB of LDS, so that six two-wave
or four four-wave workgroups share a CU.  A change to the kernel that pushes either over its budget
halves its occupancy or puts spills in the key loop, which the kernel tests would not notice (the
results stay right) but a launch runs up to a third slower."""
import os
import re
import shutil
import subprocess

import pytest

from layamd_amd import build

HIPCC = build.HIPCC


needs_hipcc = pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which(HIPCC)), reason="hipcc not available")


def _device_asm(source, tmp_path):
    """Device assembly of one source of the library, with the library's flags."""
    out = tmp_path / (source + ".s")
    flags = [f for f in build.HIP_FLAGS if f != "-fPIC"] + build.TU_FLAGS.get(source, [])
    r = subprocess.run([HIPCC] + flags + ["--cuda-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, source)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_text()


@needs_hipcc
@pytest.mark.parametrize("source", ["kernels_attn.hip", "kernels_gemm_small.hip", "kernels_norm.hip"])
def test_inline_assembly_waits_for_its_own_register_loads(source, tmp_path):
    """The compiler takes the output registers of an inline assembly block as written when the block
    ends, and may move or reuse them at once.  So a block that loads into vector registers must also
    wait for those loads: every such load is followed in its block by an s_waitcnt vmcnt(n), n no
    larger than the number of loads issued after it (LDS DMA writes no register and may stay in flight)."""
    asm = _device_asm(source, tmp_path)
    blocks = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", asm, re.S)
    for b in blocks:
        later, waited = 0, True                            # loads issued after the last register load; are those complete
        for line in b.splitlines():
            line = line.split(";")[0].strip()
            if re.match(r"(global|buffer|flat|scratch)_load", line):
                if not line.endswith(" lds"):
                    later, waited = 0, False
                else:
                    later += 1
            wait = re.match(r"s_waitcnt .*vmcnt\((\d+)\)", line)
            if wait and int(wait.group(1)) <= later:
                waited = True
        assert waited, b


def _kernels(asm):
    """(name, total VGPRs, spilled registers, scratch bytes, LDS bytes) of every kernel of the assembly."""
    val = lambda b, key: int(re.search(r"\.?" + key + r":\s+(\d+)", b).group(1))
    for b in re.split(r"\n  - ", asm[asm.index("amdhsa.kernels:"):])[1:]:
        name = re.search(r"\.name:\s+(\S+)", b)
        if name and "vgpr_count" in b:
            yield (name.group(1), val(b, "vgpr_count"), val(b, "vgpr_spill_count") + val(b, "sgpr_spill_count"),
                   val(b, "private_segment_fixed_size"), val(b, "group_segment_fixed_size"))


@needs_hipcc
def test_few_tile_and_few_row_kernels_fit_their_occupancy(tmp_path):
    """What the launch rules of the small kernels rest on: no spills; three k_attention_narrow workgroups a CU
    (160 KB of LDS; 16 queries a wave, so 3 or 6 waves a SIMD within 512 / 3 or 512 / 6 registers); two
    k_attention_f32 workgroups of 4 waves a CU when they split keys, four of whole tiles; k_gemm_small with
    one workgroup a CU in bf16, two in fp32 but for its smallest tile (32x16: a grid of at most one a CU)."""
    lds = 160 * 1024
    found = {"narrow": 0, "f32": 0, "small": 0}
    for name, vgpr, spill, scratch, l in _kernels(_device_asm("kernels_attn.hip", tmp_path)):
        if "k_attention_narrow" in name:
            found["narrow"] += 1
            assert (spill, scratch) == (0, 0) and 3 * l <= lds and vgpr <= (80 if "ILi8E" in name else 168), (name, vgpr, l)
        elif "k_attention_f32" in name:
            found["f32"] += 1
            n = 2 if "ILb1E" in name else 4
            assert (spill, scratch) == (0, 0) and n * l <= lds and vgpr <= 512 // n, (name, vgpr, l)
    for name, vgpr, spill, scratch, l in _kernels(_device_asm("kernels_gemm_small.hip", tmp_path)):
        if "k_gemm_small" in name:
            found["small"] += 1
            n = 1 if "IfLi" not in name or "Li32ELi16E" in name else 2
            assert (spill, scratch) == (0, 0) and n * l <= lds and vgpr <= 256, (name, vgpr, l)
    # bf16 tiles x epilogues, plain and split: stores and residuals of five tiles (unsplit: four), QKV of three,
    # GeGLU of two; fp32: stores and residuals of four tiles, QKV and GeGLU of two
    assert found == {"narrow": 4, "f32": 2, "small": 2 * 5 + 2 * 4 + 3 + 2 + 2 * 4 + 2 * 2}, found


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which(HIPCC)), reason="hipcc not available")
def test_attention_kernels_fit_their_occupancy(tmp_path):
    out = tmp_path / "attn.s"
    src = os.path.join(build.CSRC, "kernels_attn.hip")
    flags = [f for f in build.HIP_FLAGS if f != "-fPIC"] + build.TU_FLAGS.get("kernels_attn.hip", [])
    r = subprocess.run([HIPCC] + flags + ["--cuda-device-only", "-S", "-o", str(out), src],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    meta = out.read_text()
    # the amdhsa.kernels metadata: one block per kernel, .name after the segment sizes
    blocks = re.split(r"\n  - \.", meta[meta.index("amdhsa.kernels:"):])
    seen = {}
    for b in blocks:
        name = re.search(r"\.name:\s+(\S+)", b)
        if not name or "k_attention_bf16" not in name.group(1):
            continue
        nw = 2 if "ILi2E" in name.group(1) else 4
        val = lambda key: int(re.search(r"\." + key + r":\s+(\d+)", b).group(1))
        seen[nw] = (val("vgpr_count"), val("vgpr_spill_count"), val("group_segment_fixed_size"))
    assert set(seen) == {2, 4}, seen
    vgpr, spill, lds = seen[2]
    assert vgpr <= 168 and spill == 0 and lds == 24576, seen[2]
    vgpr, spill, lds = seen[4]
    assert vgpr <= 128 and spill <= 1 and lds == 24576, seen[4]
