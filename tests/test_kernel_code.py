"""The gfx950 code built from this repository's sources: properties that the
kernels' results or speed rest on and that only the compiler's output shows."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

LLVM = "/opt/rocm/llvm/bin"
EM_AMDGPU = 0xE0


def _code_objects():
    """The device ELF files inside libmemphys_hip.so (one per source file)."""
    import memphys_amd as M
    if not os.path.exists(M.HIP_LIB_PATH):
        import __graft_entry__ as g
        g.build()
    with open(M.HIP_LIB_PATH, "rb") as f:
        lib = f.read()
    out = []
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", lib):
        at = m.start() + 24
        (n,) = struct.unpack_from("<Q", lib, at)
        at += 8
        for _ in range(n if n < 16 else 0):
            off, size, idlen = struct.unpack_from("<QQQ", lib, at)
            at += 24 + idlen
            elf = lib[m.start() + off:m.start() + off + size]
            if elf[:4] == b"\x7fELF" and struct.unpack_from("<H", elf, 18)[0] == EM_AMDGPU:
                out.append(elf)
    assert len(out) >= 10
    return out


def _kernels(elf):
    """{symbol: metadata} of a code object's kernels (its AMDGPU note, msgpack)."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phsize)
        if kind != 4:  # PT_NOTE
            continue
        at = off
        while at < off + size:
            nlen, dlen, typ = struct.unpack_from("<III", elf, at)
            data = at + 12 + (nlen + 3) // 4 * 4
            if elf[at + 12:at + 18] == b"AMDGPU" and typ == 32:
                meta = msgpack.unpackb(elf[data:data + dlen], strict_map_key=False)
                return {k[".name"]: k for k in meta["amdhsa.kernels"]}
            at = data + (dlen + 3) // 4 * 4
    return {}


def masked_readlanes(asm):
    """Readlane instructions of a disassembled kernel in the stretches of code that
    run masked fmas with a scalar operand (from an s_and_saveexec to the next
    change of the execution mask, or to the jump back to unmasked code)."""
    total = reads = fmas = 0
    masked = False
    for line in asm.splitlines() + ["s_mov_b64 exec, -1"]:
        op = line.split("//")[0].split()
        if not op:
            continue
        if ("saveexec" in op[0] or op[0] in ("s_branch", "s_endpgm") or
                (len(op) > 1 and op[1].rstrip(",") == "exec")):
            if masked and fmas:
                total += reads
            masked, reads, fmas = "saveexec" in op[0], 0, 0
        elif op[0].startswith("v_readlane"):
            reads += 1
        elif op[0].startswith("v_fma_f64") and any(o.startswith("s[") for o in op[3:]):
            fmas += 1
    return total


def test_masked_readlanes_counts_only_masked_code():
    ok = """
	v_readlane_b32 s10, v1, s2      // 000: 0
	s_and_saveexec_b64 s[8:9], vcc
	v_fma_f64 v[0:1], v[2:3], s[10:11], v[4:5]
	s_or_b64 exec, exec, s[8:9]
	v_readlane_b32 s11, v1, s2
	s_and_saveexec_b64 s[8:9], vcc
	v_mov_b32_e32 v2, v3
"""
    assert masked_readlanes(ok) == 0
    planted = ok.replace("\tv_fma_f64", "\tv_readlane_b32 s12, v6, s2\n\tv_fma_f64")
    assert masked_readlanes(planted) == 1


@pytest.mark.parametrize("rows", [32, 48, 64])
def test_single_wavefront_weights_read_lanes_unmasked(tmp_path, rows):
    """The one-wavefront weight kernels broadcast the pivot row with readlane.
    The pivot's lane takes no part in the update, so a readlane inside the
    update's mask reads registers that the compiler need not keep for it."""
    found = 0
    for elf in _code_objects():
        for name in _kernels(elf):
            if f"weights_wave_kernelILi1ELi{rows}E" not in name:
                continue
            found += 1
            path = tmp_path / "k.elf"
            path.write_bytes(elf)
            asm = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn",
                                  f"--disassemble-symbols={name}", str(path)],
                                 check=True, capture_output=True, text=True).stdout
            assert asm.count("v_readlane") > 4 * rows  # (the broadcasts are in it)
            assert masked_readlanes(asm) == 0
    assert found == 1


@pytest.mark.parametrize("kernel", ["weights_mixed_kernel", "weights_fp64_kernel"])
def test_lds_weight_kernels_keep_eight_wavefronts(kernel):
    """The weight kernels that hold their systems in LDS hide its latency with
    eight wavefronts per SIMD: at most 64 vector registers, none spilled."""
    k, = [v for elf in _code_objects() for n, v in _kernels(elf).items() if kernel in n]
    assert k[".vgpr_count"] <= 64
    assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0
