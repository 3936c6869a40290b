"""What the machine code of the built library keeps to.

Wait states: gfx950 asks for two between a vector instruction that writes a scalar register -- a comparison's mask, a readlane, a carry
-- and a vector instruction that reads it.  The compiler sees to it for its own instructions, but not for those of inline assembly, whose
operands may come straight from such an instruction.

Scratch: kernels that are held to a number of registers fit into it.

Hints: the first pass of a transform in place stores without the non-temporal hint, which costs it up to 4 %."""
import os
import re
import struct
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT_STATES = 2

SCALAR = re.compile(r"\bs(\d+)\b|\bs\[(\d+):(\d+)\]|\b(vcc)(?:_lo|_hi)?\b")
# (operands in front of the first source; which of them may be a scalar register is for SCALAR to say)
WRITER = re.compile(r"v_(?:(?P<one>cmp_|readlane_|readfirstlane_)|(?:(?:add|sub|subrev|addc|subb|subbrev)_co_|div_scale_|mad_[iu]64_))")
IMPLICIT_VCC = re.compile(r"v_(?:cndmask_b32_e32|(?:addc|subb|subbrev)_co_u32_e32|div_fmas_)")


def _scalars(operands):
    regs = set()
    for first, low, high, vcc in SCALAR.findall(operands):
        regs |= {vcc} if vcc else ({int(first)} if first else set(range(int(low), int(high) + 1)))
    return regs


def hazards(listing):
    """(writer, reader) of every pair of vector instructions, in the order they lie in, with less than WAIT_STATES between them and a
    scalar register of the one read by the other"""
    found, recent = [], []                  # of the last instructions that wrote scalars: wait states since, registers, text
    for line in listing:
        if line[:1] != "\t":                # a label: another kernel, or a block of it (which may still follow the last one)
            continue
        op, _, rest = line.strip().partition(" ")
        states = 1
        if op == "s_nop":
            states += int(rest.split()[0], 0)
        elif op in ("s_endpgm", "s_branch", "s_setpc_b64"):
            recent = []
        elif op.startswith("v_"):
            writes = WRITER.match(op)
            if recent or writes:
                operands = rest.split("//")[0].split(", ")
                results = 2 if writes and not writes["one"] else 1
                if recent:
                    reads = _scalars(" ".join(operands[results:])) | ({"vcc"} if IMPLICIT_VCC.match(op) else set())
                    found += [(text, line.strip()) for _, regs, text in recent if regs & reads]
                if writes:
                    regs = _scalars(" ".join(operands[:results]))
                    recent = [(since + 1, r, text) for since, r, text in recent if since + 1 < WAIT_STATES]
                    if regs:
                        recent.append((0, regs, line.strip()))
                    continue
        if recent:
            recent = [(since + states, r, text) for since, r, text in recent if since + states < WAIT_STATES]
    return found


def _code_objects(lib):
    data = open(lib, "rb").read()
    at = data.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        entry = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if size and b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(BUNDLE, at + 1)


def test_the_rule_on_short_listings():
    def of(*lines):
        return len(hazards("\t" + line for line in lines))
    cmp, use = "v_cmp_lt_i64_e64 s[2:3], 0, v[2:3]", "v_cndmask_b32_e64 v5, 0, v5, s[2:3]"
    assert of(cmp, use) == of(cmp, "s_nop 0", use) == of(cmp, "v_mov_b32_e32 v1, v2", use) == 1
    assert of(cmp, "s_nop 1", use) == of(cmp, "v_mov_b32_e32 v1, v2", "s_add_u32 s9, s9, 1", use) == 0
    assert of(cmp, "v_cndmask_b32_e64 v5, 0, v5, s[4:5]") == of(cmp, "s_endpgm", use) == 0
    assert of("v_readlane_b32 s46, v41, 0", "v_readlane_b32 s47, v41, 16", "v_cndmask_b32_e64 v2, v2, -v2, s[46:47]") == 2
    assert of("v_cmp_gt_f32_e32 vcc, v1, v2", "v_cndmask_b32_e32 v1, v2, v3, vcc") == 1
    assert of("v_add_co_u32_e32 v1, vcc, v1, v2", "v_addc_co_u32_e32 v3, vcc, 0, v3, vcc") == 1


def test_vector_instructions_wait_for_scalar_registers(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    from dynamiq_sigcomm_artifact_amd import capi

    def of_object(index_code):
        path = tmp_path / ("%d.co" % index_code[0])
        path.write_bytes(index_code[1])
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], stdout=subprocess.PIPE, text=True) as p:
            found = hazards(p.stdout)
        assert p.returncode == 0
        return found

    with ThreadPoolExecutor(8) as pool:
        of_objects = list(pool.map(of_object, enumerate(_code_objects(capi.LIB_PATH))))
    assert of_objects
    found = [pair for pairs in of_objects for pair in pairs]
    assert not found, (len(found), found[:4])


def test_the_first_pass_in_place_stores_without_a_hint(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    from dynamiq_sigcomm_artifact_amd import capi
    stores = {}
    for k, code in enumerate(c for c in _code_objects(capi.LIB_PATH) if b"rht_first_kernel" in c):
        path = tmp_path / ("%d.co" % k)
        path.write_bytes(code)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], stdout=subprocess.PIPE, text=True, check=True).stdout
        for kernel in re.split(r"^[0-9a-f]+ <", listing, flags=re.M):
            name = re.match(r"\S*rht_first_kernelILb([01])E", kernel)
            if name:
                found = re.findall(r"^\t(global_store_dword\w* .*?)\s*(?://|$)", kernel, re.M)
                stores.setdefault(name[1] == "1", []).append((len(found), sum(" nt" in store for store in found)))
    assert set(stores) == {False, True}
    assert all(count > 0 and hinted == 0 for count, hinted in stores[False]), stores
    assert all(hinted > 0 for _, hinted in stores[True]), stores


def test_statistics_of_all_ranks_fit_their_registers(tmp_path):
    """ranks_stats_kernel is held to 64 registers: every variant, with and without the words of short rings, without scratch"""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    from dynamiq_sigcomm_artifact_amd import capi
    code = next(c for c in _code_objects(capi.LIB_PATH) if b"ranks_stats_kernel" in c)
    path = tmp_path / "single_pass.co"
    path.write_bytes(code)
    notes = subprocess.run([READELF, "--notes", str(path)], stdout=subprocess.PIPE, text=True, check=True).stdout
    scratch = {}
    for kernel in notes.split("- .agpr_count")[1:]:
        field = dict(re.findall(r"^\s+\.(name|private_segment_fixed_size):\s+(\S+)", kernel, re.M))
        scratch[field["name"]] = int(field["private_segment_fixed_size"])
    stats = {name: size for name, size in scratch.items() if "ranks_stats_kernel" in name}
    assert len(stats) >= 6 and not any(stats.values()), stats


def test_short_rings_leave_room_for_eight_waves(tmp_path):
    """ring_parts_kernel with four elements per lane and drawn values: 64 vector and 80 scalar registers, no scratch"""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    from dynamiq_sigcomm_artifact_amd import capi
    path = tmp_path / "single_pass.co"
    path.write_bytes(next(c for c in _code_objects(capi.LIB_PATH) if b"ring_parts_kernel" in c))
    notes = subprocess.run([READELF, "--notes", str(path)], stdout=subprocess.PIPE, text=True, check=True).stdout
    fields = [dict(re.findall(r"^\s+\.(name|private_segment_fixed_size|vgpr_count|sgpr_count):\s+(\S+)", text, re.M))
              for text in notes.split("- .agpr_count")[1:]]
    fours = [f for f in fields if re.search(r"ring_parts_kernelILi\dELi3ELb[01]ELi4E", f["name"])]
    assert len(fours) == 8, fields
    for f in fours:
        assert int(f["private_segment_fixed_size"]) == 0 and int(f["vgpr_count"]) <= 64 and int(f["sgpr_count"]) <= 80, f
