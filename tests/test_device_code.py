"""What only the machine code of the built library shows.  Distances between instructions that the compiler
keeps for its own but not for inline assembly: a v_permlane32_swap must come at least two wait
states after the vector instruction that writes one of its operands (an instruction in between counts
one, s_nop N counts N + 1).  And waits that it does not place: where a transfer behind a barrier overwrites
the LDS that was read before it, no read may be outstanding at the barrier."""
import os
import re
import struct
import subprocess

import pytest

from mace_amd import lib as mh

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """the gfx950 code objects of a host library: the entries of its offload bundles"""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n].decode()
            pos += 24 + n
            if size and name.endswith("gfx950"):
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, pos)


def registers(operand):
    """the vector registers that an operand names"""
    m = re.fullmatch(r"[va](\d+)|[va]\[(\d+):(\d+)\]", operand)
    if not m:
        return set()
    first, last = (int(m[1]),) * 2 if m[1] else (int(m[2]), int(m[3]))
    return {(operand[0], r) for r in range(first, last + 1)}


def too_close(listing, wait=2):
    """(swaps seen, [(kernel, writer, swap)]) over a disassembly; a jump's target counts as reached
    from the line above it"""
    swaps, bad, kernel, recent = 0, [], "", []   # recent: (text, registers written, wait states passed since)
    for line in listing.splitlines():
        label = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if label:
            kernel, recent = label[1], []
            continue
        text = line.split("//")[0].strip()
        if not text or line[0] not in "\t ":
            continue
        op, _, rest = text.partition(" ")
        operands = [o.strip() for o in rest.split(",")]
        if op.startswith("v_permlane32_swap"):
            swaps += 1
            read = registers(operands[0]) | registers(operands[1])
            bad += [(kernel, w, text) for w, regs, since in recent if since < wait and regs & read]
        passed = int(operands[0], 0) + 1 if op == "s_nop" else 1
        recent = [(w, regs, since + passed) for w, regs, since in recent if since + passed < wait]
        if op.startswith("v_") and not op.startswith(("v_cmp", "v_readfirstlane", "v_readlane", "v_mfma")):
            written = registers(operands[0])
            if op.startswith("v_permlane32_swap"):
                written |= registers(operands[1])
            recent.append((text, written, 0))
    return swaps, bad


RING = re.compile(r"q8_gemm_dma_kernelI")


def transfers_at_barriers(listing):
    """{ring kernel: [memory operations outstanding at each of its barriers]}; vmcnt(N) leaves N"""
    found, kernel, out = {}, None, 0
    for line in listing.splitlines():
        label = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if label:
            kernel, out = label[1] if RING.search(label[1]) else None, 0
            continue
        text = line.split("//")[0].strip()
        if kernel is None:
            continue
        if re.match(r"(buffer|global)_load", text):
            out += 1
        elif text.startswith("s_waitcnt"):
            left = re.search(r"vmcnt\((\d+)\)", text)
            out = min(out, int(left[1])) if left else out
        elif text.startswith("s_barrier"):
            found.setdefault(kernel, []).append(out)
    return found


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs ROCm's llvm-objdump")
def test_no_transfer_is_outstanding_where_the_epilogue_takes_its_lds(tmp_path):
    kernels = {}
    for i, blob in enumerate(code_objects(mh.LIB_PATH)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(blob)
        kernels.update(transfers_at_barriers(subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True,
                                                            capture_output=True, text=True).stdout))
    assert len(kernels) >= 50 and all(len(v) >= 3 for v in kernels.values()), kernels   # prologue, loop, epilogue
    assert not any(n for v in kernels.values() for n in v[2:]), {k: v for k, v in kernels.items() if any(v[2:])}


# the ring kernel with slabs of 128 bytes: its transfers refill the stage of the slab being multiplied
REFILLS = re.compile(r"q8_gemm_dma_kernelI(Li\d+E){5}[hi]Li\d+E(Lb[01]E){2}Li128E")


def reads_at_barriers(listing):
    """{kernel: [LDS reads outstanding at each of its barriers]} of the kernels that REFILLS names, in the order of the
    listing; LDS reads return in order, lgkmcnt(N) leaves N"""
    found, kernel, out = {}, None, 0
    for line in listing.splitlines():
        label = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if label:
            kernel, out = label[1] if REFILLS.search(label[1]) else None, 0
            continue
        text = line.split("//")[0].strip()
        if kernel is None:
            continue
        if text.startswith("ds_read"):
            out += 1
        elif text.startswith("s_waitcnt"):
            left = re.search(r"lgkmcnt\((\d+)\)", text)
            out = min(out, int(left[1])) if left else out
        elif text.startswith("s_barrier"):
            found.setdefault(kernel, []).append(out)
    return found


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs ROCm's llvm-objdump")
def test_no_lds_read_is_outstanding_where_its_stage_is_refilled(tmp_path):
    name = "q8_gemm_dma_kernelILi2ELi2ELi2ELi2ELi2EhLi2ELb1ELb0ELi128E"
    head, read, wait, barrier = "0000000000001000 <%s>:\n" % name, "\tds_read_b128 v[0:3], v4\n", \
        "\ts_waitcnt vmcnt(0) lgkmcnt(%d)\n", "\ts_barrier\n"
    assert reads_at_barriers(head + read + read + wait % 1 + barrier + wait % 0 + barrier) == {name: [1, 0]}
    kernels = {}
    for i, blob in enumerate(code_objects(mh.LIB_PATH)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(blob)
        kernels.update(reads_at_barriers(subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True,
                                                        capture_output=True, text=True).stdout))
    assert len(kernels) >= 20 and all(len(v) >= 3 for v in kernels.values()), kernels   # prologue, loop, epilogue
    assert not any(n for v in kernels.values() for n in v), {k: v for k, v in kernels.items() if any(v)}


def test_the_check_itself():
    head = "0000000000001000 <k>:\n"
    pack, swap = "\tv_ashr_pk_u8_i32 v4, v1, v2, s3   // 00: 00\n", "\tv_permlane32_swap_b32_e32 v5, v4   // 00: 00\n"
    other, nop = "\tv_add_u32_e32 v9, v8, v7\n", "\ts_nop %d\n"
    for between, count in (("", 1), (other, 1), (nop % 0, 1), (nop % 1, 0), (other + other, 0), (nop % 0 + other, 0)):
        assert [len(r) if isinstance(r, list) else r for r in too_close(head + pack + between + swap)] == [1, count]
    assert not too_close(head + pack.replace("v4", "v6") + swap)[1]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs ROCm's llvm-objdump")
def test_half_wave_swaps_wait_for_their_operands(tmp_path):
    mh.load()   # (builds nothing: the library is there or this fails)
    objects = list(code_objects(mh.LIB_PATH))
    assert objects
    swaps = 0
    for i, blob in enumerate(objects):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(blob)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True, capture_output=True,
                                 text=True).stdout
        seen, bad = too_close(listing)
        swaps += seen
        assert not bad, (len(bad), bad[:4])
    assert swaps > 100
