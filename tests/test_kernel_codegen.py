"""What the compiler made of the dense tile kernel's K loop, checked on the assembly (no GPU needed: hipcc cross-compiles), and the
registers that the instances of the mid-size kernel take in the built library.

The four-wavefront dense kernel runs one wavefront per SIMD, so its speed rests on properties of the generated loop that
no numerical test sees: all 256 accumulators stay in their accumulation registers across the loop (small changes to the
source have made the register allocator move them through vector registers every iteration, 14 % slower with identical
results), the loop is fully unrolled (128 matrix instructions per K step, two steps per iteration), and nothing spills.

The counts below are those of ROCm 7.2's hipcc on the source as committed.  Another compiler version may schedule or
allocate differently without anything being wrong with the kernel: a failure here after a toolchain change alone means
"measure the dense kernel again" (bench.py, gemm.roofline), not "the kernel is broken".
"""
import os
import re
import shutil
import struct
import subprocess

import pytest

from sensenova_u1_amd import build


def _assembly(tmp_path, src):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    out = tmp_path / (os.path.splitext(src)[0] + ".s")
    cmd = [hipcc, *build.HIP_FLAGS, *build.SOURCE_FLAGS.get(src, []), "-x", "hip", "-S", "--cuda-device-only",
           os.path.join(build.CSRC, src), "-o", str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    return out.read_text()


def test_dense_kernel_loop_keeps_its_accumulators_in_place(tmp_path):
    text = _assembly(tmp_path, "gemm_dense4.hip")
    lines = text.splitlines()
    starts = [i for i, l in enumerate(lines) if re.match(r"^_ZN6sngguf.*gemm_dense4_kernelILi\dEEE.*:", l)]
    assert len(starts) == 4, "one kernel instance per epilogue"
    for s in starts:
        name = lines[s].split(":")[0]
        end = next(i for i in range(s, len(lines)) if lines[i].startswith(".Lfunc_end"))
        # basic blocks of the function: the K loop is the one with the most matrix instructions
        blocks, cur = [], []
        for l in lines[s:end]:
            if re.match(r"^\.LBB\d+_\d+:", l):
                blocks.append(cur)
                cur = []
            cur.append(l)
        blocks.append(cur)
        loop = max(blocks, key=lambda b: sum("v_mfma_f32_16x16x32_bf16" in l for l in b))
        count = lambda pat: sum(bool(re.search(pat, l)) for l in loop)
        assert count(r"v_mfma_f32_16x16x32_bf16") == 256, name          # two K steps of 128, fully unrolled
        assert count(r"v_accvgpr_(read|write|mov)") == 0, name           # accumulators stay where they are
        assert count(r"\bds_read_b128\b") == 64, name                    # 16 fragments per half step
        assert count(r"global_load_lds_dwordx4") == 32, name             # 16 copies per step
        assert count(r"scratch_(load|store)") == 0, name
    for field in ("vgpr_spill_count", "sgpr_spill_count", "private_segment_fixed_size"):
        vals = re.findall(rf"\.{field}:\s+(\d+)", text)
        assert vals and all(v == "0" for v in vals), (field, vals)


def _kernel_resources(tmp_path):
    """{kernel symbol: its metadata's numbers} over the device code objects that the built library holds."""
    readelf = "/opt/rocm/llvm/bin/llvm-readelf"
    if not os.path.exists(readelf) or not os.path.exists(build.LIB_PATH):
        pytest.skip("llvm-readelf or the built library not found")
    with open(build.LIB_PATH, "rb") as f:
        lib = f.read()
    magic, pos, found, objects = b"__CLANG_OFFLOAD_BUNDLE__", -1, {}, 0
    while (pos := lib.find(magic, pos + 1)) >= 0:   # magic, count, then (offset, size, length of the target's name, name) each
        count, at = struct.unpack_from("<Q", lib, pos + len(magic))[0], pos + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", lib, at)
            target = lib[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" not in target or size == 0:
                continue
            obj = tmp_path / f"object{objects}"
            objects += 1
            obj.write_bytes(lib[pos + offset:pos + offset + size])
            notes = subprocess.run([readelf, "--notes", str(obj)], capture_output=True, text=True).stdout
            for name, body in re.findall(r"\.name: +(\S+)\n(.*?)\.wavefront_size", notes, re.S):
                found[name] = {f: int(v) for f, v in re.findall(r"\.(\w+): +(\d+)\n", body)}
    return found


def _mid_instances(tmp_path):
    """{(format, numerics, row groups, 16-row tiles, K shares, ...): numbers} of gemm_mid_kernel."""
    out = {}
    for name, numbers in _kernel_resources(tmp_path).items():
        m = re.search(r"gemm_mid_kernelI((?:L[ib]\d+E)+)E", name)
        if m:
            out[tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1)))] = numbers
    return out


def test_mid_size_kernel_does_not_spill(tmp_path):
    """Spilled registers of the K loop cost up to a quarter of the time and change no result."""
    instances = _mid_instances(tmp_path)
    assert len(instances) >= 260
    assert {k: v["vgpr_spill_count"] for k, v in instances.items() if v["vgpr_spill_count"] or v["private_segment_fixed_size"]} == {}


def test_mid_size_kernel_leaves_room_for_two_workgroups(tmp_path):
    """Eight wavefronts of at most 128 registers fit a compute unit twice, which launches of more than 256 workgroups count on: the
    narrow form, and the wide form of 32 and 48 rows in the formats whose decode is small enough."""
    wide = {2: {2, 3, 6, 7, 8, 10, 11, 12}, 3: {2, 3, 7, 10, 12}}   # 16-row tiles: ggml types
    too_many = {}
    for (qt, _, groups, tiles, *_), numbers in (instances := _mid_instances(tmp_path)).items():
        if (groups == 1 or qt in wide.get(tiles, ())) and numbers["vgpr_count"] > 128:
            too_many[qt, groups, tiles] = numbers["vgpr_count"]
    assert instances and too_many == {}
